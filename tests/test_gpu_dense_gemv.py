"""Dense single-vector products at the edges of their tiles: rows and columns
around the 16-byte runs, the wavefront's rows, the column slabs and the
one-, two- and four-column wavefronts of A^T x.  Compared with FP64 products
of the stored matrix; tolerance: the FP32 (FP64) summation bound
K u |A| |x| with u = 2^-24 (2^-53) for sums of K terms."""
import numpy as np
import pytest

from tval3_amd import api

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import torch
    assert torch.cuda.is_available()
    return api.Context(0)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16", "f64"])
@pytest.mark.parametrize("m,n", [(1, 1), (3, 5), (7, 70), (8, 64), (255, 9), (257, 130), (512, 65),
                                 (519, 33), (1030, 513), (65, 4097), (77, 8195)])
def test_gemv_edges(ctx, m, n, dtype):
    import torch
    rng = np.random.default_rng(m * 10007 + n)
    A = np.asfortranarray(rng.normal(size=(m, n)).astype(np.float32))
    op = api.DenseOperator(ctx, A, dtype)
    stored = {"f32": A, "f64": A, "f16": A.astype(np.float16),
              "bf16": torch.from_numpy(A).bfloat16().float().numpy()}[dtype].astype(np.float64)
    vt, u = (np.float64, 2.0 ** -53) if dtype == "f64" else (np.float32, 2.0 ** -24)
    for trans, M in ((False, stored), (True, stored.T)):
        # one element into a longer buffer: vectors need not be 16-byte aligned
        x = rng.normal(size=M.shape[1] + 1).astype(vt)
        y = op.mat_vec_mul(torch.from_numpy(x).cuda()[1:], trans=trans).cpu().numpy()
        x = x[1:].astype(np.float64)
        bound = (M.shape[1] + 2) * u * (np.abs(M) @ np.abs(x))
        assert (np.abs(y - M @ x) <= bound).all(), (trans, np.abs(y - M @ x).max())
