"""Performance cases: the work users of this framework have it do, through its
public entry points (tval3_amd.api, tval3_amd.autograd).

Kinds of work:

* ``sparse``  a ray matrix given as CSR arrays, y = A x and z = A^T r, for one
  vector (mat_vec_mul) or several (mat_mat_mul);
* ``dense``   the same for a dense matrix;
* ``rays``    the same for a transducer geometry, the weights generated inside
  the product (Siddon lengths or Bresenham walks);
* ``tv``      one total-variation layer of the autograd binding, forward and
  backward: V = D u, W = shrink(V), q = D^T (V - W);
* ``solve``   a whole TVAL3 solve with a fixed number of inner iterations.

Geometry: transducers on a sphere of radius 1.1 around the volume [-1, 1]^3,
every emitter with every receiver, as in the benchmark and the tests.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "tval3-gpu_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from tval3_amd import api, autograd as ad  # noqa: E402

_DEV = "cuda"
_BYTES = {"f32": 4, "f16": 2, "bf16": 2, "f64": 8}


def listed():
    return [
        # the smallest call: an operator test or a toy volume, latency only
        dict(name="sparse_f32_tiny", kind="sparse", p=12, q=12, r=12, E=24, R=48, dtype="f32",
             nrhs=1),
        # the benchmark's matrix (128^3 voxels, 262,144 rays) with FP16 weights,
        # used through the operator plug-in
        dict(name="sparse_f16_128", kind="sparse", p=128, q=128, r=128, E=256, R=1024,
             dtype="f16", nrhs=1),
        # several measurement vectors over one FP32 matrix of 64^3 voxels
        dict(name="sparse_f32_64_rhs8", kind="sparse", p=64, q=64, r=64, E=128, R=512,
             dtype="f32", nrhs=8),
        # a 64 x 64 image from 1,638 dense measurements
        dict(name="dense_f32_1638x4096", kind="dense", m=1638, n=4096, dtype="f32", nrhs=1),
        # a dense operator of 32 x 32 x 16 voxels with BF16 weights, one vector
        dict(name="dense_bf16_8192x16384", kind="dense", m=8192, n=16384, dtype="bf16", nrhs=1),
        # problems sharing that dense operator: 64 right-hand sides
        dict(name="dense_bf16_4096x16384_rhs64", kind="dense", m=4096, n=16384, dtype="bf16",
             nrhs=64),
        # matrix-free Siddon products at 96^3 (192 emitters, 768 receivers)
        dict(name="siddon_96", kind="rays", mode="siddon", p=96, q=96, r=96, E=192, R=768,
             dtype="f32"),
        # the same on a volume cut to odd sizes
        dict(name="siddon_ragged", kind="rays", mode="siddon", p=77, q=101, r=90, E=150, R=601,
             dtype="f32"),
        # the reference's own ray model (integer walks) at 128^3
        dict(name="bresenham_128", kind="rays", mode="bresenham", p=128, q=128, r=128, E=256,
             R=1024, dtype="f32"),
        # a total-variation layer inside a training step, 96^3
        dict(name="tv_f32_96", kind="tv", p=96, q=96, r=96, dtype="f32", iso=True),
        # the default solver on host arrays, 64^3 voxels and 65,536 rays
        dict(name="solve_plain_f32_64", kind="solve", solver="plain", p=64, q=64, r=64, E=128,
             R=512, weights="f32", dtype="f32", iters=20, iso=True),
        # the benchmark: fused solver, FP16 weights, 128^3
        dict(name="solve_fused_f16_128", kind="solve", solver="fused", p=128, q=128, r=128,
             E=256, R=1024, weights="f16", dtype="f32", iters=20, iso=True),
    ]


# ------------------------------------------------------------------- drawing
def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _edges(rng, lo, hi):
    return tuple(_log_int(rng, lo, hi) for _ in range(3))


def _transducers(rng, lo, hi):
    """Emitters and receivers, E : R about 1 : 4, lo to hi rays in all."""
    rays = _log_int(rng, lo, hi)
    E = max(1, int(round(math.sqrt(rays) / 2 * rng.uniform(0.7, 1.4))))
    return E, max(1, min(rays // E, hi // E))


def draw(rng):
    kind = rng.choice(["sparse", "sparse", "dense", "dense", "rays", "rays", "tv", "solve"])
    if kind == "sparse":
        p, q, r = _edges(rng, 12, 128)
        nrhs = rng.choice([1, 1, 1, 2, 4, 8, 13])
        E, R = _transducers(rng, 1152, 262144 if nrhs == 1 else 65536 * 8 // (8 * nrhs))
        if nrhs > 1:
            p, q, r = min(p, 64), min(q, 64), min(r, 64)
        return dict(kind=kind, p=p, q=q, r=r, E=E, R=R,
                    dtype=rng.choice(["f32", "f16", "bf16"] + (["f64"] if nrhs == 1 else [])),
                    nrhs=nrhs)
    if kind == "dense":
        nrhs = rng.choice([1, 1, 1, 2, 8, 64])
        dtype = rng.choice(["f32", "f16", "bf16"] + (["f64"] if nrhs == 1 else []))
        if nrhs > 1 and rng.random() < 0.5:
            # whole blocks of 256, as a shared dense operator of a batch has
            return dict(kind=kind, m=256 * _log_int(rng, 2, 16), n=256 * _log_int(rng, 4, 64),
                        dtype="bf16", nrhs=nrhs)
        return dict(kind=kind, m=_log_int(rng, 200, 4096), n=_log_int(rng, 1000, 16384),
                    dtype=dtype, nrhs=nrhs)
    if kind == "rays":
        mode = rng.choice(["siddon", "bresenham"])
        p, q, r = _edges(rng, 12, 110)
        if rng.random() < 0.5:
            p, q, r = (max(12, v // 4 * 4) for v in (p, q, r))
        E, R = _transducers(rng, 1152, 147456)
        return dict(kind=kind, mode=mode, p=p, q=q, r=r, E=E, R=R,
                    dtype=rng.choice(["f32", "f32", "f32", "f64"]))
    if kind == "tv":
        p, q, r = _edges(rng, 12, 96)
        return dict(kind=kind, p=p, q=q, r=r, dtype=rng.choice(["f32", "f32", "f64"]),
                    iso=rng.random() < 0.5)
    solver = rng.choice(["plain", "plain", "fused"])
    if solver == "fused":
        p, q, r = (8 * _log_int(rng, 2, 12) for _ in range(3))
    else:
        p, q, r = _edges(rng, 12, 64)
    E, R = _transducers(rng, 1152, 65536)
    dtype = rng.choice(["f32", "f32", "f64"]) if solver == "plain" else "f32"
    weights = rng.choice(["f16", "bf16", "f32"]) if solver == "fused" else "f32"
    return dict(kind=kind, solver=solver, p=p, q=q, r=r, E=E, R=R, weights=weights, dtype=dtype,
                iters=rng.randint(5, 20), iso=rng.random() < 0.7)


# -------------------------------------------------------------------- inputs
def _dims(c):
    return c["p"], c["q"], c["r"]


def _voxels(c):
    return c["p"] * c["q"] * c["r"]


def _gen(seed, salt):
    return torch.Generator(device=_DEV).manual_seed(seed * 1009 + salt)


def _randn(seed, salt, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=_gen(seed, salt), device=_DEV, dtype=dtype)


def _phantom(c, seed):
    """Slowness: 1/1500 s/m with six ellipsoids at +/- 3 %, float64."""
    p, q, r = _dims(c)
    g = np.random.default_rng([seed, 1])
    ax = [torch.linspace(-1 + 1.0 / k, 1 - 1.0 / k, k, device=_DEV, dtype=torch.float64)
          for k in (r, q, p)]
    Z, X, Y = torch.meshgrid(*ax, indexing="ij")
    u = torch.full_like(X, 1.0 / 1500.0)
    for _ in range(6):
        cx, cy, cz = g.uniform(-0.6, 0.6, 3)
        a, b, d = g.uniform(0.08, 0.35, 3)
        inside = ((X - cx) / a) ** 2 + ((Y - cy) / b) ** 2 + ((Z - cz) / d) ** 2 <= 1.0
        u[inside] = (1.0 + 0.03 * (1 if g.uniform() < 0.5 else -1)) / 1500.0
    return u.reshape(-1)


def _geometry(c, seed):
    p, q, r = _dims(c)
    g = np.random.default_rng([seed, 2])
    pts = g.normal(size=(c["E"] + c["R"], 3))
    pts = (1.1 * pts / np.linalg.norm(pts, axis=1, keepdims=True)).astype(np.float32)
    num = np.array([q, p, r])
    voxel = (2.0 / num).astype(np.float32)
    vox = np.clip(np.floor((pts + 1.0) / voxel), 0, num - 1).astype(np.int32)
    E = c["E"]
    return dict(E=E, R=c["R"], mps=1, rv=(q, p, r), origin=(-1.0, -1.0, -1.0),
                voxel=tuple(float(v) for v in voxel), e_pos=pts[:E], r_pos=pts[E:],
                e_vox=vox[:E], r_vox=vox[E:], scale=float(voxel[0]), use_path=None)


def _trace(geom, chunk=32768):
    """Per chunk of rays: voxel index and intersection length of every piece
    of every ray, float64; pieces outside the volume have length 0."""
    num = geom["rv"]
    h = [float(v) for v in geom["voxel"]]
    ep = torch.tensor(geom["e_pos"], device=_DEV, dtype=torch.float64)
    rp = torch.tensor(geom["r_pos"], device=_DEV, dtype=torch.float64)
    R, rays = geom["R"], geom["E"] * geom["R"]
    for k0 in range(0, rays, chunk):
        k = torch.arange(k0, min(rays, k0 + chunk), device=_DEV)
        a, d = ep[k // R], rp[k % R] - ep[k // R]
        lo = torch.zeros(len(k), device=_DEV, dtype=torch.float64)
        hi = torch.ones_like(lo)
        planes = []
        for ax in range(3):
            pl = -1.0 + h[ax] * torch.arange(num[ax] + 1, device=_DEV, dtype=torch.float64)
            t = (pl[None, :] - a[:, ax:ax + 1]) / d[:, ax:ax + 1]
            lo = torch.maximum(lo, torch.minimum(t[:, 0], t[:, -1]))
            hi = torch.minimum(hi, torch.maximum(t[:, 0], t[:, -1]))
            planes.append(t)
        hi = torch.maximum(lo, hi)
        t = torch.cat(planes, 1).clamp(lo[:, None], hi[:, None]).sort(1).values
        mid, dt = (t[:, 1:] + t[:, :-1]) / 2, t[:, 1:] - t[:, :-1]
        ix = [((a[:, ax:ax + 1] + mid * d[:, ax:ax + 1] + 1.0) / h[ax]).floor().long()
              .clamp(0, num[ax] - 1) for ax in range(3)]
        yield (ix[2] * num[0] + ix[0]) * num[1] + ix[1], dt * d.norm(dim=1, keepdim=True)


def _round(v, dtype):
    """float64 values rounded to a weight type, as float64."""
    t = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16,
         "f64": torch.float64}[dtype]
    return v.float().to(t).double() if dtype != "f64" else v


def _ray_matrix(geom, dtype):
    """CSR of the Siddon matrix: row pointers, columns, weights (float64
    holding values of the weight type); device tensors."""
    cnt, col, val = [], [], []
    for v, ln in _trace(geom):
        keep = ln > 1e-7
        cnt.append(keep.sum(1))
        col.append(v[keep].int())
        val.append(_round(ln[keep], dtype))
    ptr = torch.zeros(geom["E"] * geom["R"] + 1, device=_DEV, dtype=torch.int64)
    ptr[1:] = torch.cat(cnt).cumsum(0)
    return ptr, torch.cat(col), torch.cat(val)


def _measure(geom, u, seed):
    """b = A u + 0.5 % noise, float64."""
    b = torch.cat([(u[v] * ln).sum(1) for v, ln in _trace(geom)])
    xi = torch.randn(len(b), generator=_gen(seed, 3), device=_DEV, dtype=torch.float64)
    return b + 0.005 * b.norm() * xi / xi.norm()


def _vectors(c, seed, n, m, field=True):
    """x (a volume) and r (measurements) of a product, or nrhs of each."""
    dt = torch.float64 if c["dtype"] == "f64" else torch.float32
    k = c.get("nrhs", 1)
    if field:
        x = _phantom(c, seed)[None, :] * (1 + 0.05 * torch.rand(
            k, n, generator=_gen(seed, 4), device=_DEV, dtype=torch.float64))
    else:
        x = torch.rand(k, n, generator=_gen(seed, 4), device=_DEV, dtype=torch.float64)
    r = _randn(seed, 5, k, m, dtype=torch.float64)
    x, r = x.to(dt), r.to(dt)
    return (x[0], r[0]) if k == 1 else (x.t(), r.t())


def _dense_matrix(c, seed):
    """N(0, 1/m) entries as an (n, m) tensor: column j of A is row j."""
    return _randn(seed, 6, c["n"], c["m"]) / math.sqrt(c["m"])


def _tv_inputs(c, seed):
    dt = torch.float64 if c["dtype"] == "f64" else torch.float32
    n = _voxels(c)
    u = _phantom(c, seed) * 1500.0 - 1.0 + 0.01 * _randn(seed, 7, n, dtype=torch.float64)
    gq = _randn(seed, 8, n, dtype=torch.float64)
    gs = _randn(seed, 9, n, dtype=torch.float64)
    return u.to(dt), gq.to(dt), gs.to(dt)


_TV_T = 0.02    # shrinkage threshold of the tv cases


# ------------------------------------------------------------------- the API
def prepare(case, seed):
    c, kind = case, case["kind"]
    ctx = api.Context(0)
    st = dict(case=c, ctx=ctx)
    if kind == "sparse":
        geom = _geometry(c, seed)
        ptr, col, val = _ray_matrix(geom, c["dtype"])
        st["A"] = api.SparseOperator(ctx, geom["E"] * geom["R"], _voxels(c),
                                     ptr.int().cpu().numpy(), col.cpu().numpy(),
                                     (val if c["dtype"] == "f64" else val.float()).cpu().numpy(),
                                     dtype=c["dtype"])
        st["x"], st["r"] = _vectors(c, seed, st["A"].n, st["A"].m)
    elif kind == "dense":
        A = _dense_matrix(c, seed).cpu().numpy().T
        st["A"] = api.DenseOperator(ctx, A, dtype=c["dtype"])
        st["x"], st["r"] = _vectors(c, seed, c["n"], c["m"], field=False)
    elif kind == "rays":
        st["A"] = api.DynamicOperator(ctx, _geometry(c, seed), c["mode"])
        st["x"], st["r"] = _vectors(c, seed, st["A"].n, st["A"].m)
    elif kind == "tv":
        st["u"], st["gq"], st["gs"] = _tv_inputs(c, seed)
    else:
        geom = _geometry(c, seed)
        st["A"] = api.DynamicOperator(ctx, geom, "siddon").materialize(c["weights"])
        b = _measure(geom, _phantom(c, seed), seed)
        b = b if c["dtype"] == "f64" else b.float()
        # the default solver takes host arrays, as the reference's does; the
        # fused one device tensors
        st["b"] = b.cpu().numpy() if c["solver"] == "plain" else b
        st["opts"] = api.default_opts(mu=2.0 ** 9, mu0=2.0 ** 9, maxit=c["iters"], tol=0.0,
                                      tol_inn=0.0, solver=c["solver"],
                                      tv_mode="iso" if c["iso"] else "aniso")
        if c["solver"] == "fused":
            st["A"].prepare(_dims(c))
    return st


def run(state):
    c = state["case"]
    if c["kind"] in ("sparse", "dense", "rays"):
        A = state["A"]
        if c.get("nrhs", 1) > 1:
            return [A.mat_mat_mul(state["x"]), A.mat_mat_mul(state["r"], trans=True)]
        return [A.mat_vec_mul(state["x"]), A.mat_vec_mul(state["r"], trans=True)]
    if c["kind"] == "tv":
        u = state["u"].detach().requires_grad_(True)
        ctx, dims = state["ctx"], _dims(c)
        V = ad.grad3(ctx, u, dims)
        W, s, active = ad.shrink(ctx, V, _TV_T, iso=c["iso"])
        q = ad.grad3_t(ctx, V - W, dims)
        (gu,) = torch.autograd.grad((q, s), u, (state["gq"], state["gs"]))
        return [W.detach(), s.detach(), active, q.detach(), gu]
    U, _, _ = api.tval3_gpu_3d(state["ctx"], state["A"], state["b"], _dims(c), state["opts"],
                               history=False)
    return [U]


def _entries(c):
    """Matrix entries of a ray case: about 1.07 (Siddon) or 0.67 (Bresenham)
    per ray and voxel of the mean edge."""
    per = 0.67 if c.get("mode") == "bresenham" else 1.07
    return int(per * (c["p"] + c["q"] + c["r"]) / 3 * c["E"] * c["R"])


def work(case):
    c, kind = case, case["kind"]
    v = 8 if c["dtype"] == "f64" else 4
    if kind == "dense":
        k, mn = c["nrhs"], c["m"] * c["n"]
        return {"bytes": 2 * mn * _BYTES[c["dtype"]] + 2 * k * v * (c["m"] + c["n"]),
                "flops": 4 * k * mn}
    n = _voxels(c)
    if kind == "tv":      # u, gq, gs in; W, s, active, q, gu out
        return {"bytes": 9 * v * n + n, "flops": 60 * n}
    m, nnz = c["E"] * c["R"], _entries(c)
    vec = 2 * v * (m + n)
    if kind == "rays":
        return {"bytes": vec + 24 * (c["E"] + c["R"]), "flops": 4 * nnz}
    if kind == "sparse":
        k = c["nrhs"]
        return {"bytes": 2 * nnz * (4 + _BYTES[c["dtype"]]) + 4 * (m + n) + k * vec,
                "flops": 4 * k * nnz}
    # per inner iteration one product each way and the stencil steps' streams
    # (U, g, three sigma, the multiplier term, d in; U, d, g out; U, d, Au)
    it = c["iters"] + 1
    return {"bytes": it * (2 * nnz * (4 + _BYTES[c["weights"]]) + 4 * (m + n) + vec + 15 * v * n),
            "flops": it * (4 * nnz + 100 * n)}


# --------------------------------------------------------------- 64-bit values
def _rows_of(ptr, nnz):
    return torch.repeat_interleave(torch.arange(len(ptr) - 1, device=_DEV), ptr[1:] - ptr[:-1],
                                   output_size=nnz)


class _Coo:
    """A x and A^T r of a ray matrix, float64."""

    def __init__(self, geom, n, dtype):
        ptr, col, self.val = _ray_matrix(geom, dtype)
        self.col, self.row = col.long(), _rows_of(ptr, len(col))
        self.m, self.n = len(ptr) - 1, n

    def A(self, x):
        return torch.zeros(self.m, device=_DEV, dtype=torch.float64).index_add_(
            0, self.row, self.val * x[self.col])

    def At(self, r):
        return torch.zeros(self.n, device=_DEV, dtype=torch.float64).index_add_(
            0, self.col, self.val * r[self.row])


def _walks(geom):
    """Bresenham walks: per step (ray mask, voxel index)."""
    nx, ny, nz = geom["rv"]
    e = torch.tensor(geom["e_vox"], device=_DEV).long()
    r = torch.tensor(geom["r_vox"], device=_DEV).long()
    k = torch.arange(geom["E"] * geom["R"], device=_DEV)
    c = e[k // geom["R"]].clone()
    d = r[k % geom["R"]] - c
    inc, a = torch.where(d < 0, -1, 1), d.abs()
    # leading axis: x before y before z among equals; the others in order
    lead = torch.where((a[:, 0] >= a[:, 1]) & (a[:, 0] >= a[:, 2]), 0,
                       torch.where((a[:, 1] >= a[:, 0]) & (a[:, 1] >= a[:, 2]), 1, 2))
    others = torch.tensor([[1, 2], [0, 2], [0, 1]], device=_DEV)[lead]
    al = a.gather(1, lead[:, None])
    ao = a.gather(1, others)
    err = 2 * ao - al
    for j in range(int(al.max()) + 1):
        yield al[:, 0] >= j, (c[:, 2] * nx + c[:, 0]) * ny + c[:, 1]
        up = err > 0
        c.scatter_add_(1, others, up * inc.gather(1, others))
        err = err - up * 2 * al + 2 * ao
        c.scatter_add_(1, lead[:, None], inc.gather(1, lead[:, None]))
        c = torch.minimum(c.clamp(min=0), torch.tensor([nx - 1, ny - 1, nz - 1], device=_DEV))


def _D(u, dims):
    p, q, r = dims
    v = u.reshape(r, q, p)
    return torch.stack([(v.roll(-1, ax) - v).reshape(-1) for ax in (1, 2, 0)])


def _Dt(V, dims):
    p, q, r = dims
    X, Y, Z = (t.reshape(r, q, p) for t in V)
    return ((X.roll(1, 1) - X) + (Y.roll(1, 2) - Y) + (Z.roll(1, 0) - Z)).reshape(-1)


def _shrink(V, t, iso):
    if not iso:
        s = (V.abs() - t).clamp(min=0)
        return V.sign() * s, s.sum(0)
    r = V.norm(dim=0)
    s = (r - t).clamp(min=0)
    return V * (s / torch.where(r > 0, r, torch.ones_like(r))), s


def _tval3(M, dims, b, iters, iso, mu=512.0, beta=32.0, c_armijo=1e-5, gamma=0.6, gam=0.9995,
           rate_gam=0.9):
    """TVAL3 (augmented Lagrangian, Barzilai-Borwein steps, nonmonotone line
    search) for iters inner iterations of one outer iteration."""
    lo, hi = b[b.abs().argmin()], b[b.abs().argmax()]
    dif = float((hi - lo).abs())
    scl = 0.5 / dif if dif < 0.5 else 1.5 / dif if dif > 1.5 else 1.0
    b = b * scl
    Atb = M.At(b)
    beta = min(beta, 32.0)
    mdb = mu / beta

    def split(U):                       # DU, W, lam1
        DU = _D(U, dims)
        W, s = _shrink(DU, 1.0 / beta, iso)
        return DU, W, float(s.sum())

    U = Atb.clone()
    DU, W, lam1 = split(U)
    Au = M.A(U)
    g, g2 = M.At(Au) - Atb, _Dt(DU - W, dims)

    def value(DU, W, Au, lam1):
        return lam1 + beta / 2 * float((DU - W).square().sum()) + \
            mu / 2 * float((Au - b).square().sum())

    f = value(DU, W, Au, lam1)
    d = mdb * g + g2
    Q, C, first = 1.0, f, True

    def exact_step(d):
        dd = float(d.square().sum())
        return abs(dd / (float(_D(d, dims).square().sum()) + mdb * float(M.A(d).square().sum())))

    def descend(U, tau):
        U = (U - tau * d).clamp(min=0)
        DU, Au = _D(U, dims), M.A(U)
        return U, DU, Au, M.At(Au) - Atb, _Dt(DU - W, dims)

    for _ in range(iters):
        if first:
            tau = exact_step(d)
        else:
            y = (g2 - g2p) + mdb * (g - gp)
            tau = abs(float(s.square().sum()) / float((s * y).sum()))
        Up, gp, g2p, Aup, DUp = U, g, g2, Au, DU
        U, DU, Au, g, g2 = descend(Up, tau)
        f = value(DU, W, Au, lam1)
        alpha, arm = 1.0, float(d.square().sum()) * tau * c_armijo * beta
        full = (U, DU, Au, g, g2)
        cnt = 0
        while abs(f) > abs(C - alpha * arm):
            if cnt == 5:
                gam *= rate_gam
                tau = exact_step(d)
                U, DU, Au, g, g2 = descend(Up, tau)
                f = value(DU, W, Au, lam1)
                break
            alpha *= gamma
            U, DU, Au, g, g2 = (pv + alpha * (nv - pv) for pv, nv in
                                zip((Up, DUp, Aup, gp, g2p), full))
            f = value(DU, W, Au, lam1)
            cnt += 1
        W, sh = _shrink(DU, 1.0 / beta, iso)
        lam1 = float(sh.sum())
        f = value(DU, W, Au, lam1)
        g2 = _Dt(DU - W, dims)
        Qp, Q = Q, gam * Q + 1
        C = (gam * Qp * C + f) / Q
        s = U - Up
        d = mdb * g + g2
        first = False
    return U / scl


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "dense":
        At = _round(_dense_matrix(c, seed).double(), c["dtype"])
        x, r = _vectors(c, seed, c["n"], c["m"], field=False)
        return [At.t() @ x.double(), At @ r.double()]
    if kind == "tv":
        u, gq, gs = (t.double() for t in _tv_inputs(c, seed))
        u.requires_grad_(True)
        V = _D(u, _dims(c))
        W, s = _shrink(V, _TV_T, c["iso"])
        q = _Dt(V - W, _dims(c))
        (gu,) = torch.autograd.grad((q, s), u, (gq, gs))
        return [W.detach(), s.detach(), None, q.detach(), gu]
    geom, n = _geometry(c, seed), _voxels(c)
    m = geom["E"] * geom["R"]
    if kind == "sparse":
        M = _Coo(geom, n, c["dtype"])
        x, r = (t.double() for t in _vectors(c, seed, n, m))
        if c["nrhs"] == 1:
            return [M.A(x), M.At(r)]
        return [torch.stack([M.A(v) for v in x.t()]).t(),
                torch.stack([M.At(v) for v in r.t()]).t()]
    if kind == "rays":
        x, r = (t.double() for t in _vectors(c, seed, n, m))
        if c["mode"] == "siddon":
            M = _Coo(geom, n, "f64")
            return [M.A(x), M.At(r)]
        w = float(np.float32(geom["scale"]))
        y, z = torch.zeros_like(r), torch.zeros_like(x)
        for on, v in _walks(geom):
            y += torch.where(on, x[v], 0.0)
            z.index_add_(0, v, torch.where(on, r, 0.0))
        return [w * y, w * z]
    b = _measure(geom, _phantom(c, seed), seed)
    b = b if c["dtype"] == "f64" else b.float().double()
    return [_tval3(_Coo(geom, n, c["weights"]), _dims(c), b, c["iters"], c["iso"])]
