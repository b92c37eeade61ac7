"""A x of sparse matrices whose x is larger than an XCD's L2 (more than 2^20
columns): row blocks run in the order of the columns they touch where
neighbouring blocks lie apart, else in natural order.  Whole numbers, so both
orders give the exact product; few blocks, many, an odd count, empty rows and
rows longer than a block among them."""
import numpy as np
import pytest

from tval3_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [3, 700, 20_011])
@pytest.mark.parametrize("rows", ["scattered", "local", "unstructured"])
def test_rows_in_either_order(rows, m):
    import torch
    assert torch.cuda.is_available()
    ctx = api.Context(0)
    n, width = (1 << 20) + 77, 4000
    rng = np.random.default_rng(m)
    lens = rng.integers(0, 120, m)
    lens[m // 2] = 700
    if rows == "scattered":
        first = rng.integers(0, n - width, m)
    else:
        first = np.arange(m) * (n - width) // m if rows == "local" else np.zeros(m, np.int64)
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    r = np.repeat(np.arange(m), lens)
    col = (first[r] + rng.integers(0, n if rows == "unstructured" else width, len(r))).astype(np.int32)
    val = rng.integers(-3, 4, len(col)).astype(np.float64)
    for dtype, vec in (("f16", np.float32), ("f32", np.float64)):
        op = api.SparseOperator(ctx, m, n, rowptr, col, val, dtype=dtype)
        x = rng.integers(-4, 5, (3, n)).astype(vec)
        want = np.stack([np.bincount(r, val * v[col], minlength=m) for v in x])
        xd = torch.from_numpy(x).cuda()
        for j in range(3):
            assert (op.mat_vec_mul(xd[j]).cpu().numpy() == want[j]).all(), (dtype, j)
        if vec is np.float32:
            assert (op.mat_mat_mul(xd.t()).cpu().numpy() == want.T).all()
