"""Products in flight on several streams at once (two; five, more than have a
workspace of their own), of one operator and of several operators of a context:
every result equals the one computed alone, bit for
bit.  Dense products share the context's partial sums, the matrix-core
products the operator's copies as well."""
import numpy as np
import pytest

from tval3_amd import api, workload as wl

pytestmark = pytest.mark.gpu


def _check(calls):
    """Runs calls alone, then from stream to stream."""
    import torch
    want = [f() for f in calls]
    torch.cuda.synchronize()
    for count in (2, 5):
        streams = [torch.cuda.Stream() for _ in range(count)]
        got = []
        for k in range(5 * len(calls)):
            with torch.cuda.stream(streams[k % count]):
                got.append(calls[k % len(calls)]())
        torch.cuda.synchronize()
        for k, y in enumerate(got):
            assert torch.equal(y, want[k % len(calls)]), (count, k)


def _cols(n, k, seed, dtype=None):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(k, n, device="cuda", generator=g, dtype=dtype).t()


@pytest.mark.parametrize("dtype,m,n", [("f32", 2047, 4093), ("bf16", 1000, 9000), ("f64", 900, 3000)])
def test_dense(dtype, m, n):
    import torch
    assert torch.cuda.is_available()
    ctx = api.Context(0)
    rng = np.random.default_rng(m)
    ops = [api.DenseOperator(ctx, np.asfortranarray(rng.normal(size=(m + d, n)).astype(np.float32)),
                             dtype) for d in (0, 64)]
    vec = torch.float64 if dtype == "f64" else torch.float32
    xs = [_cols(n, 1, s, vec)[:, 0].contiguous() for s in range(3)]
    calls = [lambda op=op, x=x: op.mat_vec_mul(x) for x in xs for op in ops]
    if dtype != "f64":
        X = _cols(n, 8, 9)
        calls += [lambda op=op: op.mat_mat_mul(X) for op in ops]
    _check(calls)


def test_matrix_core_products():
    import torch
    assert torch.cuda.is_available()
    ctx = api.Context(0)
    A = np.random.default_rng(3).normal(size=(1024, 4096)).astype(np.float32)
    op = api.DenseOperator(ctx, np.asfortranarray(A), "bf16")
    X, R, x = _cols(4096, 64, 1), _cols(1024, 64, 2), _cols(4096, 1, 3)[:, 0].contiguous()
    _check([lambda: op.mat_mat_mul(X), lambda: op.mat_mat_mul(R, trans=True),
            lambda: op.mat_vec_mul(x)])


def test_matrix_core_first_product_on_each_stream():
    # the operand copies are made by the first product, on its stream
    import torch
    assert torch.cuda.is_available()
    ctx = api.Context(0)
    A = np.random.default_rng(4).integers(-3, 4, (2048, 8192)).astype(np.float32)
    op = api.DenseOperator(ctx, np.asfortranarray(A), "bf16")
    X = torch.randint(-4, 5, (64, 8192), device="cuda").float().t()
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s1):
        a = op.mat_mat_mul(X)
    with torch.cuda.stream(s2):
        b = op.mat_mat_mul(X)
    torch.cuda.synchronize()
    want = torch.from_numpy(A).cuda().double() @ X.double()
    assert torch.equal(a.double(), want) and torch.equal(b.double(), want)


def _tiles(ctx):
    # 32^3 voxels, 16,384 rays: tile products of some 20 us
    return api.DynamicOperator(ctx, wl.transducer_geometry(64, 256, dims=(32, 32, 32), seed=3),
                               "siddon")


def test_siddon_tiles():
    import torch
    assert torch.cuda.is_available()
    op = _tiles(api.Context(0))
    xs = [_cols(op.n, 1, s)[:, 0].contiguous() for s in range(3)]
    rs = [_cols(op.m, 1, s)[:, 0].contiguous() for s in range(3)]
    _check([lambda x=x: op.mat_vec_mul(x) for x in xs] +
           [lambda r=r: op.mat_vec_mul(r, trans=True) for r in rs])
    # without an allocation: one call after the other, the same bits
    for x, r in zip(xs, rs):
        for v, trans in ((x, False), (r, True)):
            y = torch.empty(op.n if trans else op.m, device="cuda")
            op.mat_vec_mul_noalloc(v, y, trans=trans)
            assert torch.equal(y, op.mat_vec_mul(v, trans=trans))


def test_siddon_tiles_beside_a_solve_and_a_graph():
    import torch
    assert torch.cuda.is_available()
    ctx = api.Context(0)
    op = _tiles(ctx)
    x, r = _cols(op.n, 1, 1)[:, 0].contiguous(), _cols(op.m, 1, 2)[:, 0].contiguous()
    b = np.linspace(0.5, 1.5, op.m).astype(np.float32)
    o = api.default_opts(maxit=4, tol=0.0, tol_inn=0.0, solver="fused")
    want = op.mat_vec_mul(x), op.mat_vec_mul(r, trans=True)
    U = api.tval3_gpu_3d(ctx, op, b, (32, 32, 32), o)[0]
    y, z = torch.zeros_like(want[0]), torch.zeros_like(want[1])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        op.mat_vec_mul(x, y)
        op.mat_vec_mul(r, z, trans=True)
    other = torch.cuda.Stream()
    for k in range(4):
        y.zero_()
        z.zero_()
        torch.cuda.synchronize()
        for _ in range(5):
            graph.replay()
        with torch.cuda.stream(other):
            got = [(op.mat_vec_mul(x), op.mat_vec_mul(r, trans=True)) for _ in range(20)]
        assert (api.tval3_gpu_3d(ctx, op, b, (32, 32, 32), o)[0] == U).all(), k
        torch.cuda.synchronize()
        for g in got + [(y, z)]:
            assert torch.equal(g[0], want[0]) and torch.equal(g[1], want[1]), k
