"""The workspace of dense products A X: what the launch's column slabs need,
and products recorded into a graph, whatever ran before.  A graph is replayed
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


def test_graph_keeps_its_workspace():
    # eager products, larger ones too, on the replaying stream and on another
    # while a graph's products are in flight; a second graph whose products
    # need a larger workspace.  Random values: the eager product's bits.
    import torch
    assert torch.cuda.is_available()
    ctx = api.Context(0)
    rng = np.random.default_rng(5)
    small, large = (api.DenseOperator(ctx, np.asfortranarray(
        rng.normal(size=(m, n)).astype(np.float32)), "f32") for m, n in ((700, 3000), (1500, 9000)))
    g = torch.Generator(device="cuda").manual_seed(1)
    xs, xl = (torch.randn(8, n, device="cuda", generator=g).t() for n in (3000, 9000))
    ys, yl = small.mat_mat_mul(xs), large.mat_mat_mul(xl)
    outs, outl = torch.zeros_like(ys), torch.zeros_like(yl)
    torch.cuda.synchronize()
    graphs = []
    for op, x, y in ((small, xs, outs), (large, xl, outl)):
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1]):
            op.mat_mat_mul(x, y)
    other = torch.cuda.Stream()
    for k in range(4):
        outs.zero_()
        outl.zero_()
        torch.cuda.synchronize()
        graphs[0].replay()
        graphs[1].replay()
        with torch.cuda.stream(other):
            a = large.mat_mat_mul(xl)
        b = small.mat_mat_mul(xs)
        torch.cuda.synchronize()
        for got, want in ((outs, ys), (outl, yl), (a, yl), (b, ys)):
            assert torch.equal(got, want), k
