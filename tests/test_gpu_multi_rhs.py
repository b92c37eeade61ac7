"""Products of several vectors (mat_mat_mul) where the matrix cores do not
serve: every column equals mat_vec_mul of that column bit for bit (the same
additions in the same order), at the edges of the column tiles, for rows
longer than a block, empty rows, every row-block size, and the row-group
kernel; also when two streams use one operator."""
import numpy as np
import pytest

from tval3_amd import api

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import torch
    assert torch.cuda.is_available()
    return api.Context(0)


def _cols(n, k, seed, pad=0):
    """(n, k) float32 tensor, columns contiguous, leading dimension n + pad"""
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(k, n + pad, device="cuda", generator=g)[:, :n].t()


def _sparse(ctx, dtype):
    rng = np.random.default_rng(31)
    m, n = 900, 9000
    lens = np.concatenate([[0, 5000, 3, 0, 4100, 1200], rng.integers(0, 60, m - 6)])
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(n, l, replace=False)) for l in lens]).astype(np.int32)
    return api.SparseOperator(ctx, m, n, rowptr, col, rng.normal(size=len(col)), dtype=dtype)


def _check(op, nrhs, seed):
    import torch
    for trans in (False, True):
        X = _cols(op.m if trans else op.n, nrhs, seed, pad=3)
        Y = op.mat_mat_mul(X, trans=trans)
        for j in range(nrhs):
            y = op.mat_vec_mul(X[:, j].contiguous(), trans=trans)
            assert torch.equal(Y[:, j], y), (trans, j)


@pytest.mark.parametrize("nrhs", [1, 2, 3, 4, 5, 8, 9, 13])
@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
def test_sparse_columns_equal_matvec(ctx, dtype, nrhs):
    op = _sparse(ctx, dtype)
    for code in (-2048, -1024, -4096, 8):
        op.set_lanes(code, code)
        _check(op, nrhs, nrhs)


@pytest.mark.parametrize("nrhs", [2, 3, 4, 5, 8, 11])
@pytest.mark.parametrize("dtype,m,n", [("f32", 6, 40), ("f32", 519, 301), ("f16", 130, 4099),
                                       ("bf16", 1027, 513), ("bf16", 300, 8200)])
def test_dense_columns_equal_matvec(ctx, dtype, m, n, nrhs):
    A = np.random.default_rng(m).normal(size=(m, n)).astype(np.float32)
    _check(api.DenseOperator(ctx, np.asfortranarray(A), dtype), nrhs, nrhs)


def test_sparse_on_two_streams(ctx):
    import torch
    op = _sparse(ctx, "f32")
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    X = [_cols(op.n, 8, s) for s in range(6)]
    want = [op.mat_mat_mul(x) for x in X]
    torch.cuda.synchronize()
    got = []
    for k, x in enumerate(X):
        with torch.cuda.stream((s1, s2)[k % 2]):
            got.append(op.mat_mat_mul(x))
    torch.cuda.synchronize()
    for w, y in zip(want, got):
        assert torch.equal(w, y)
