"""Matrix-core products whose K splits are not of equal lengths: one chunk of
64 values, fewer chunks than splits would like, prime numbers of chunks.
Against FP64 products of the same BF16 matrix, elementwise within
4 sqrt(K) 2^-24 |A||X| (three BF16 terms of X, FP32 accumulation)."""
import numpy as np
import pytest

from tval3_amd import api

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import torch
    assert torch.cuda.is_available()
    return api.Context(0)


@pytest.mark.parametrize("m,n", [(256, 64), (256, 192), (512, 448), (768, 1216), (2304, 832),
                                 (256, 8128), (1280, 5376)])
@pytest.mark.parametrize("nrhs", [5, 64])
def test_uneven_splits_against_fp64(ctx, m, n, nrhs):
    import torch
    g = torch.Generator(device="cuda").manual_seed(m + n)
    A = torch.randn(m, n, generator=g, device="cuda").bfloat16().double()
    op = api.DenseOperator(ctx, np.asfortranarray(A.cpu().numpy()), dtype="bf16")
    for trans, M in ((False, A), (True, A.t())):
        X = torch.randn(nrhs, M.shape[1], generator=g, device="cuda").t()
        Y = op.mat_mat_mul(X, trans=trans).double()
        err = (Y - M @ X.double()).abs()
        bound = 4 * np.sqrt(M.shape[1]) * 2.0 ** -24 * (M.abs() @ X.double().abs())
        assert (err <= bound).all(), (trans, (err / bound).max().item())
