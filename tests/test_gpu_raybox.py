"""Matrix-free products outside the tile layout (Bresenham, FP64, volumes
with dimensions that are not multiples of 4): A x per ray, A^T r from the
rays' parts inside boxes of 16 x 8 x 8 voxels.  Compared with the matrix the
device materializes from the same traversal (pinned to the oracle by
test_gpu_ops.py and test_gpu_dyntile.py), in FP64; tolerance: the summation
bound K u |A| |x|, u = 2^-24 (2^-53 for FP64), for K terms and their products.
Shapes: volumes smaller than a box, box remainders along every axis, boxes
whose segments are split over several workgroups, masked rays, two
measurement positions, and transducers outside the grid (clamped walks)."""
import numpy as np
import pytest

from tval3_amd import api, workload as wl

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import torch
    assert torch.cuda.is_available()
    return api.Context(0)


def _two_positions(E, R, dims):
    a, b = (wl.transducer_geometry(E, R, dims=dims, seed=s) for s in (5, 6))
    return dict(a, mps=2, **{k: np.concatenate([a[k], b[k]])
                             for k in ("e_pos", "r_pos", "e_vox", "r_vox")})


def _masked(E, R, dims):
    return dict(wl.transducer_geometry(E, R, dims=dims, seed=7),
                use_path=(np.arange(E * R) % 3 != 1).astype(np.uint8))


def _outside(E, R, dims):
    g = wl.transducer_geometry(E, R, dims=dims, seed=8)
    return dict(g, e_vox=g["e_vox"] - 3, r_vox=g["r_vox"] + 2)


GEOMS = {
    "tiny": lambda: wl.transducer_geometry(3, 5, dims=(5, 3, 2), seed=2),
    "remainders": lambda: wl.transducer_geometry(20, 45, dims=(17, 9, 23), seed=3),
    "long_y": lambda: wl.transducer_geometry(9, 64, dims=(61, 7, 8), seed=4),
    "split_boxes": lambda: wl.transducer_geometry(96, 256, dims=(16, 13, 10), seed=9),
    # Siddon on 8^3 tiles of about 26,000 entries: A^T boxes of half a tile
    "half_tiles": lambda: wl.transducer_geometry(48, 256, dims=(16, 16, 16), seed=2),
    "two_positions": lambda: _two_positions(10, 30, (22, 18, 15)),
    "masked": lambda: _masked(24, 40, (19, 21, 33)),
    "outside": lambda: _outside(12, 24, (20, 14, 11)),
}


@pytest.mark.parametrize("dt", ["f32", "f64"])
@pytest.mark.parametrize("mode", ["bresenham", "siddon"])
@pytest.mark.parametrize("name", list(GEOMS))
def test_products_equal_materialized_matrix(ctx, name, mode, dt):
    import torch
    op = api.DynamicOperator(ctx, GEOMS[name](), mode)
    rp, col, val = op.materialize("f32").download_csr()
    row = np.repeat(np.arange(op.m), np.diff(rp))
    vt, u = (np.float64, 2.0 ** -53) if dt == "f64" else (np.float32, 2.0 ** -24)
    rng = np.random.default_rng(1)
    x = rng.uniform(-1, 1, size=op.n).astype(vt)
    r = rng.normal(size=op.m).astype(vt)
    r[::7] = 0
    for trans, vec, out, src, size in ((False, x, row, col, op.m), (True, r, col, row, op.n)):
        y = op.mat_vec_mul(torch.from_numpy(vec).cuda(), trans=trans).cpu().numpy()
        terms = val * vec[src].astype(np.float64)
        want = np.bincount(out, terms, size)
        bound = np.bincount(out, np.abs(terms), size)
        k = np.bincount(out, minlength=size).max() + 2
        err = np.abs(y - want)
        assert (err <= k * u * bound).all(), (trans, err.max())


@pytest.mark.parametrize("mode", ["bresenham", "siddon"])
@pytest.mark.parametrize("E,R", [(1, 1), (256, 255), (256, 256), (512, 257), (512, 512)])
def test_lanes_sharing_a_ray(ctx, E, R, mode):
    # A x with 8, 4, 2 and 1 lanes a ray (by the number of rays), walks shorter
    # than the lanes are many
    import torch
    op = api.DynamicOperator(ctx, wl.transducer_geometry(E, R, dims=(13, 6, 9), seed=11), mode)
    rp, col, val = op.materialize("f32").download_csr()
    rng = np.random.default_rng(E + R)
    x = rng.normal(size=op.n).astype(np.float32)
    rows = np.repeat(np.arange(op.m), np.diff(rp))
    t = val.astype(np.float64) * x[col]
    want = np.bincount(rows, t, minlength=op.m)
    mass = np.bincount(rows, np.abs(t), minlength=op.m)
    k = np.diff(rp) + 2
    y = op.mat_vec_mul(torch.from_numpy(x).cuda()).cpu().numpy()
    assert (np.abs(y - want) <= k * 2.0 ** -24 * mass).all()
