"""A new sparse operator's products: one wavefront per row block of 256
entries, a longer row by itself, workgroup blocks where a row has more than
4096 entries.  Whole numbers, so every product is exact whatever the order of
its additions; rows at the blocks' edges (255, 256, 257, 512, 4096, 4097
entries), empty rows, and more short rows than a block has lanes."""
import numpy as np
import pytest

from tval3_amd import api

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import torch
    assert torch.cuda.is_available()
    return api.Context(0)


LENGTHS = {
    "short": [0] * 70 + [1] * 200 + [0, 3, 0] * 50 + [2] * 65,
    "edge256": [255, 1, 256, 0, 1, 255, 256, 128, 129] + [4] * 64 + [256],
    "edge512": [257, 255, 512, 0, 1, 511, 512, 300, 213] + [8] * 64 + [512],
    "long": [513, 5, 0, 2048, 1, 3000, 4096] + [7] * 300,
    "longer": [513, 4097, 0, 2048, 1, 3000, 4096] + [7] * 300,
    "one": [6],
}


def _matrix(name):
    rng = np.random.default_rng(41)
    lens = np.array(LENGTHS[name])
    m, n = len(lens), 4100
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(n, l, replace=False)) for l in lens]).astype(np.int32)
    val = rng.integers(-3, 4, len(col)).astype(np.float64)
    A = np.zeros((m, n))
    A[np.repeat(np.arange(m), lens), col] = val
    return A, rowptr, col, val


@pytest.mark.parametrize("name", list(LENGTHS))
@pytest.mark.parametrize("dtype,vec", [("f32", "float32"), ("f16", "float32"), ("bf16", "float32"),
                                       ("f32", "float64"), ("f64", "float64")])
def test_default_blocks_exact(ctx, name, dtype, vec):
    import torch
    A, rowptr, col, val = _matrix(name)
    # A^T's rows are A's columns, so both directions see every length
    for M, (rp, c, v) in ((A, (rowptr, col, val)), (A.T, _csr(A.T))):
        op = api.SparseOperator(ctx, M.shape[0], M.shape[1], rp, c, v, dtype=dtype)
        for trans, B in ((False, M), (True, M.T)):
            X = np.random.default_rng(7).integers(-4, 5, (3, B.shape[1])).astype(vec)
            Xd = torch.from_numpy(X).cuda()
            for j in range(3):
                y = op.mat_vec_mul(Xd[j], trans=trans)
                assert (y.cpu().numpy() == B @ X[j]).all(), (trans, j)
            if vec == "float32":
                Y = op.mat_mat_mul(Xd.t(), trans=trans)
                assert (Y.cpu().numpy() == B @ X.T).all(), trans


def _csr(M):
    r, c = np.nonzero(M)
    rp = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=M.shape[0]))]).astype(np.int32)
    return rp, c.astype(np.int32), M[r, c]


@pytest.mark.parametrize("name", ["edge256", "edge512", "long", "longer"])
@pytest.mark.parametrize("nrhs", [2, 4, 5, 8, 11])
def test_default_blocks_columns_equal_matvec(ctx, name, nrhs):
    import torch
    A, rowptr, col, _ = _matrix(name)
    op = api.SparseOperator(ctx, A.shape[0], A.shape[1], rowptr, col,
                            np.random.default_rng(5).normal(size=len(col)))
    g = torch.Generator(device="cuda").manual_seed(nrhs)
    for trans in (False, True):
        X = torch.randn(nrhs, op.m if trans else op.n, device="cuda", generator=g).t()
        Y = op.mat_mat_mul(X, trans=trans)
        for j in range(nrhs):
            assert torch.equal(Y[:, j], op.mat_vec_mul(X[:, j].contiguous(), trans=trans)), (trans, j)


@pytest.mark.parametrize("n", [1 << 20, (1 << 20) + 1, 3_000_000])
def test_block_order_exact(ctx, n):
    # more columns than an L2 slice holds: blocks run in another order than the
    # rows'; empty rows, and columns at both ends
    import torch
    rng = np.random.default_rng(n)
    lens = np.concatenate([[0, 300, 1, 0], rng.integers(0, 90, 900), [0, 257]])
    m = len(lens)
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    col = rng.integers(0, n, rowptr[-1]).astype(np.int32)
    col[[0, -1]] = n - 1, 0
    val = rng.integers(-3, 4, len(col)).astype(np.float32)
    op = api.SparseOperator(ctx, m, n, rowptr, col, val, dtype="f16")
    x = rng.integers(-4, 5, (2, n)).astype(np.float32)
    rows = np.repeat(np.arange(m), lens)
    want = np.stack([np.bincount(rows, val * v[col], minlength=m) for v in x])
    xd = torch.from_numpy(x).cuda()
    assert (op.mat_vec_mul(xd[0]).cpu().numpy() == want[0]).all()
    assert (op.mat_mat_mul(xd.t()).cpu().numpy() == want.T).all()
