"""A host solve that refuses b (NaN, Inf) leaves no copy of the caller's arrays
queued: the context's stream, busy when the call starts, is idle when it
returns.  The arrays are pinned, so that copies of them are asynchronous."""
import numpy as np
import pytest

from tval3_amd import _lib as L, api, workload as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver,vec", [("plain", "float32"), ("plain", "float64"),
                                        ("fused", "float32")])
@pytest.mark.parametrize("bad", [np.nan, -np.inf])
def test_stream_is_idle_after_refusal(solver, vec, bad):
    import torch
    assert torch.cuda.is_available()
    ctx = api.Context(0)
    dims = (16, 16, 16)
    A = api.DynamicOperator(ctx, wl.transducer_geometry(24, 64, dims=dims, seed=1),
                            "siddon").materialize("f32")
    dt = getattr(torch, vec)
    b = torch.linspace(0.5, 1.5, A.m, dtype=dt).pin_memory().numpy()
    Ut = torch.ones(A.n, dtype=dt).pin_memory().numpy()
    o = api.default_opts(maxit=2, solver=solver)
    stream = torch.cuda.ExternalStream(ctx.stream)
    M = torch.rand(8192, 8192, device="cuda")
    out = torch.empty_like(M)
    torch.mm(M, M, out=out)
    api.tval3_gpu_3d(ctx, A, b, dims, o, Ut=Ut)          # allocations are done
    b[A.m // 2] = bad
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        for _ in range(20):                              # some 100 ms of work
            torch.mm(M, M, out=out)
    assert not stream.query()
    with pytest.raises(L.TV3Error):
        api.tval3_gpu_3d(ctx, A, b, dims, o, Ut=Ut)
    assert stream.query()
