"""A fused layout that is built without timing its launch shapes
(layout_force on an operator that was not prepared, a code of 0 keeping what
the layout came with): products on whole numbers against the oracle's, bit for
bit, launch codes that layout_force takes back, and a solve that agrees with a
timed layout's over its first iterations."""
import numpy as np
import pytest

import tv3_oracle as orc
from tval3_amd import api, workload as wl

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import torch
    assert torch.cuda.is_available()
    return api.Context(0)


@pytest.mark.parametrize("kw", [{}, dict(code_N=-1024, panels=1), dict(code_N=16),
                                dict(code_T=-2048, panels=2)])
@pytest.mark.parametrize("dims", [(16, 16, 16), (12, 10, 6)])
def test_untimed_layout_products_exact(ctx, dims, kw):
    import torch
    dyn = api.DynamicOperator(ctx, wl.transducer_geometry(24, 64, dims=dims, seed=1), "siddon")
    rp, c, _ = dyn.materialize("f32").download_csr()
    w = (1 + (np.arange(len(c)) * 2654435761 % 7)).astype(np.float64)
    op = api.SparseOperator(ctx, dyn.m, dyn.n, rp, c, w, dtype="f16")
    info = op.layout_force(dims, **kw)
    assert info["panels"] == kw.get("panels", 0)
    again = op.layout_force(dims, info["code_N"], info["code_T"], 16384, info["panels"])
    assert (again["code_N"], again["code_T"]) == (info["code_N"], info["code_T"])
    oop = orc.csr_op(op.m, op.n, rp, c, w)
    rng = np.random.default_rng(7)
    for trans, k in ((0, op.n), (1, op.m)):
        x = rng.integers(0, 1024, k).astype(np.float32)
        want = orc.matvec(oop, trans, x.astype(np.float64)).astype(np.float32)
        got = op.layout_mat_vec_mul(dims, torch.from_numpy(x).cuda(), trans=bool(trans))
        assert (got.cpu().numpy() == want).all(), trans


def test_untimed_layout_solve(ctx):
    dims = (16, 16, 16)
    geom = wl.transducer_geometry(24, 64, dims=dims, seed=1)
    dyn = api.DynamicOperator(ctx, geom, "siddon")
    A, B = dyn.materialize("f32"), dyn.materialize("f32")
    b = orc.matvec(orc.csr_op(A.m, A.n, *A.download_csr()), 0, wl.phantom_3d(16, 3))
    A.layout_force(dims)
    o = api.default_opts(maxit=5, tol=0.0, tol_inn=0.0, mu=2.0 ** 9, mu0=2.0 ** 9, solver="fused")
    h = [api.tval3_gpu_3d(ctx, op, b.astype(np.float32), dims, o)[2] for op in (A, B)]
    # FP32 sums in another order, as the fused solver's tests bound them
    assert np.allclose(h[0]["f"][:4], h[1]["f"][:4], rtol=1e-5)
