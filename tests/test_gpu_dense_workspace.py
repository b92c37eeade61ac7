"""The workspace of dense products A X: what the launch's column slabs need,
and products recorded into a graph, where it cannot grow.  A graph is replayed
several times with eager products between, every replay compared."""
import numpy as np
import pytest

from tval3_amd import api

pytestmark = pytest.mark.gpu


def _dense(ctx, m, n, dtype="f32"):
    A = np.random.default_rng(m + n).integers(-3, 4, (m, n)).astype(np.float32)
    return api.DenseOperator(ctx, np.asfortranarray(A), dtype), A


def _ints(shape, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(-4, 5, shape, device="cuda", generator=g).float()


def test_workspace_is_what_the_slabs_need():
    # 32768 rows fill the chip with at most 8 slabs of the 16 that 1024 columns
    # allow: five vectors need at most 8 x 5 x 32768 floats (5.2 MB; device
    # memory is taken in units of at most 2 MiB).  A product of another context
    # comes first: loading its kernels takes memory too.
    import torch
    assert torch.cuda.is_available()
    other, ctx = api.Context(0), api.Context(0)
    m, n = 32768, 1024
    _dense(other, 400, 900)[0].mat_mat_mul(_ints((5, 900), 1).t())
    op, _ = _dense(ctx, m, n)
    X, Y = _ints((5, n), 1).t(), _ints((5, m), 2).t()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    op.mat_mat_mul(X, Y)
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] <= 8 * 5 * m * 4 + (2 << 20)


@pytest.mark.parametrize("first", ["nothing", "one", "eight"])
@pytest.mark.parametrize("m,n,dtype", [(300, 5000, "f32"), (1000, 777, "bf16"), (3, 900, "f16")])
def test_products_under_capture(m, n, dtype, first):
    # whole numbers: exact in any number of slabs
    import torch
    assert torch.cuda.is_available()
    ctx = api.Context(0)
    op, A = _dense(ctx, m, n, dtype)
    X, x = _ints((11, n), 3).t(), _ints((n,), 4)
    Y, y = torch.zeros(11, m, device="cuda").t(), torch.zeros(m, device="cuda")
    if first == "one":
        op.mat_vec_mul(x)
    elif first == "eight":
        op.mat_mat_mul(X[:, :8])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        op.mat_mat_mul(X, Y)
        op.mat_vec_mul(x, y)
    A = torch.from_numpy(A).cuda().double()
    for k in range(4):
        X.copy_(_ints((11, n), 10 + k).t())
        x.copy_(_ints((n,), 20 + k))
        Y.zero_()
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(Y.double(), (A @ X.double())) and torch.equal(y.double(), A @ x.double()), k
        torch.cuda.synchronize()
