// dynamic.hip -- matrix-free ray operators: ray-path weights are generated
// inside every product (geom_mm_multGPU / dyn_calc_kernel of the reference,
// 3d/mat_vec_mul_dynamic.h:682-967, 3d/tval3_gpu_3d_kernels.cu:1612-1764).
//
// Two weight modes:
//  * BRESENHAM -- the reference's integer 3-D walk from the emitter voxel to
//    the receiver voxel, constant weight scale_factor per visited voxel
//    (3d/tval3_gpu_3d_kernels.cu:1656-1759); coordinates are clamped into the
//    grid for both N and T (the reference clamps N through its texture,
//    :2167-2170, and does not check T).
//  * SIDDON -- exact intersection lengths of the emitter->receiver segment
//    with the voxel grid (Siddon, Med. Phys. 12(2), 1985), traversed in
//    increasing ray parameter by tracking the next plane of every axis
//    (siddon.hpp).
//
// FP32 products of a Siddon operator whose dimensions are multiples of 4
// run as tile products (dyntile.hip, panels.hpp: deterministic, no
// atomics).  The others -- Bresenham, FP64, other shapes -- run here.  N: one
// thread walks one ray and gathers x along it, several gathers in flight.  T:
// the rays' parts inside boxes of 16 x 8 x 8 voxels, listed on the device at
// creation (RayBoxes), add into the box in LDS; nothing is scattered to
// memory.  Neither keeps scratch between calls.  A Bresenham operator with
// transducers outside the grid keeps the clamping per-ray kernels.  The same
// walk, with FP
// contraction disabled, fills the CSR in dynamic_materialize so a
// precomputed matrix holds exactly the weights the dynamic product uses.
#include <algorithm>
#include <cmath>
#include <numeric>

#include "panels.hpp"

namespace tv3 {

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// Bresenham walk; emit(x, y, z) for each visited voxel (not clamped).
template <typename F>
__device__ __forceinline__ void bresenham_steps(int x0, int y0, int z0, int x1, int y1, int z1,
                                                F emit) {
    int c[3] = {x0, y0, z0};
    emit(c[0], c[1], c[2]);
    int d1 = x1 - x0, d2 = y1 - y0, d3 = z1 - z0;
    int m1 = abs(d1), m2 = abs(d2), m3 = abs(d3);
    int a1, a2, a3;
    if (m1 >= m2 && m1 >= m3) {
        a1 = 0; a2 = 1; a3 = 2;
    } else if (m2 >= m1 && m2 >= m3) {
        int t = d1; d1 = d2; d2 = t;
        a1 = 1; a2 = 0; a3 = 2;
    } else {
        int t = d1; d1 = d3; d3 = d2; d2 = t;
        a1 = 2; a2 = 0; a3 = 1;
    }
    int inc1 = d1 < 0 ? -1 : 1, inc2 = d2 < 0 ? -1 : 1, inc3 = d3 < 0 ? -1 : 1;
    m1 = abs(d1); m2 = abs(d2); m3 = abs(d3);
    int e1 = 2 * m2 - m1, e2 = 2 * m3 - m1;
    for (int j = 1; j < m1 + 1; ++j) {
        if (e1 > 0) { c[a2] += inc2; e1 -= 2 * m1; }
        if (e2 > 0) { c[a3] += inc3; e2 -= 2 * m1; }
        e1 += 2 * m2; e2 += 2 * m3;
        c[a1] += inc1;
        emit(c[0], c[1], c[2]);
    }
}

// The walk clamped into the grid; emit(linear voxel index).
template <typename F>
__device__ __forceinline__ void bresenham_walk(int x0, int y0, int z0, int x1, int y1, int z1,
                                               int rvx, int rvy, int rvz, F emit) {
    bresenham_steps(x0, y0, z0, x1, y1, z1, [&](int x, int y, int z) {
        emit((int64_t)clampi(z, 0, rvz - 1) * rvx * rvy + (int64_t)clampi(x, 0, rvx - 1) * rvy +
             clampi(y, 0, rvy - 1));
    });
}

// A Bresenham walk that can start at any step (transducers inside the grid).
// After j steps the leading axis has moved j voxels and a slower one, with
// differences m along it and M along the leading axis, floor((2 m j + M - 1)
// / (2 M)): its error term passes 0 that often.  off advances by the strides
// the caller gives; with all coordinates below 2^15 every term fits 32 bits.
struct BresWalk {
    int off, s1, s2, s3;     // offset, signed strides along the leading and slower axes
    int e1, e2, d1, d2, dm;  // error terms, 2 m2, 2 m3, 2 M
    int x, y, z, steps;      // voxel at the start; steps of the whole walk
    __device__ __forceinline__ BresWalk(const int4 w, int j0, int sx, int sy, int sz) {
        const int dx = w.y >> 16, dy = (int)(int16_t)w.z, dz = w.z >> 16;
        const int mx = abs(dx), my = abs(dy), mz = abs(dz);
        const int ix = dx < 0 ? -1 : 1, iy = dy < 0 ? -1 : 1, iz = dz < 0 ? -1 : 1;
        const int lead = mx >= my && mx >= mz ? 0 : (my >= mx && my >= mz ? 1 : 2);
        const int M = lead == 0 ? mx : (lead == 1 ? my : mz);
        const int m2 = lead == 0 ? my : mx, m3 = lead == 2 ? my : mz;
        d1 = 2 * m2; d2 = 2 * m3; dm = 2 * M;
        int k2 = 0, k3 = 0;
        if (j0 > 0) {        // then M > 0
            k2 = (int)((unsigned)(d1 * j0 + M - 1) / (unsigned)dm);
            k3 = (int)((unsigned)(d2 * j0 + M - 1) / (unsigned)dm);
        }
        e1 = d1 * (j0 + 1) - M - dm * k2;
        e2 = d2 * (j0 + 1) - M - dm * k3;
        x = (int)(int16_t)w.x + ix * (lead == 0 ? j0 : k2);
        y = (w.x >> 16) + iy * (lead == 1 ? j0 : (lead == 0 ? k2 : k3));
        z = (int)(int16_t)w.y + iz * (lead == 2 ? j0 : k3);
        sx *= ix; sy *= iy; sz *= iz;
        s1 = lead == 0 ? sx : (lead == 1 ? sy : sz);
        s2 = lead == 0 ? sy : sx;
        s3 = lead == 2 ? sy : sz;
        off = 0;
        steps = M + 1;
    }
    __device__ __forceinline__ void next() {
        const bool a = e1 > 0, b = e2 > 0;
        off += s1 + (a ? s2 : 0) + (b ? s3 : 0);
        e1 += d1 - (a ? dm : 0);
        e2 += d2 - (b ? dm : 0);
    }
};

// Siddon traversal of p0->p1 through [org, org + N*h] (siddon.hpp);
// emit(linear voxel index, length) in traversal order.
template <typename R, typename F>
__device__ __forceinline__ void siddon_walk(const R p0[3], const R p1[3], const R org[3],
                                            const R h[3], const int N[3], int rvy_stride, F emit) {
    SidRay<R> s;
    sid_setup(s, p0, p1, org, h, N);
    if (!s.hit) return;
    sid_walk(s, s.amin, s.amax, [&](int cx, int cy, int cz, R w) {
        emit((int64_t)cz * N[0] * rvy_stride + (int64_t)cx * rvy_stride + cy, w);
    });
}

struct GeoView {
    int32_t rvx, rvy, rvz;
    float scale;
    const int32_t *path, *ec, *rc;
    const float *ep, *rp;
    float org[3], h[3];
    int64_t P;
};

static GeoView view(const DynGeom &g) {
    GeoView v;
    v.rvx = g.rv_x; v.rvy = g.rv_y; v.rvz = g.rv_z;
    v.scale = g.scale;
    v.path = g.path.p; v.ec = g.ecoord.p; v.rc = g.rcoord.p;
    v.ep = g.epos.p; v.rp = g.rpos.p;
    for (int a = 0; a < 3; ++a) { v.org[a] = g.origin[a]; v.h[a] = g.voxel[a]; }
    v.P = g.num_paths;
    return v;
}

// Boxes of the A^T product (RayBoxes) and its workgroup.  Measured, Bresenham
// at 128^3 and Siddon at 77 x 101 x 90 (us): 16 x 8 x 8 voxels, 512 threads,
// items of at most 8192 segments 44, 27; 4096 segments 51, 27; 256 threads
// and 4096 52, 28; 8^3 voxels 55, 25; 16^3 voxels 60-67, 34-44.
constexpr int kRayBoxY = 16, kRayBoxXZ = 8, kBoxThreads = 512;
constexpr int kBoxSegs = 8192, kLenClasses = 16;

template <typename R>
__device__ __forceinline__ void ray_ends(const GeoView &g, int64_t k, R p0[3], R p1[3]) {
    int e = g.path[2 * k], r = g.path[2 * k + 1];
#pragma unroll
    for (int a = 0; a < 3; ++a) { p0[a] = (R)g.ep[3 * e + a]; p1[a] = (R)g.rp[3 * r + a]; }
}

// N of a Bresenham operator with every transducer in the grid: 1 << lg lanes
// share a ray's steps, one behind the other (rays in bundles of neighbours, so
// the lanes of a wavefront gather near each other), and gather eight voxels at
// a time; one at a time, each step waited for its gather.  At 128^3 with
// 262,144 rays 206 -> 77 us, now bound by the lines of the gathers: 19.6M L1
// accesses (0.4 a clock and CU), 13.5M of them on to L2 (22 TB/s; vector issue
// takes 13 us).  4 to 32 at a time, bundles of 4^2 to 32^2 rays and workgroups
// of 64 to 1024 threads all take 77-79 us; x in bricks of 4 x 4 x 2 voxels 70,
// and 6 for the copy.
template <typename T, typename AccT>
__global__ __launch_bounds__(64) void k_bres_N(GeoView g, const int32_t *__restrict__ bundle,
                                               const int4 *__restrict__ walk,
                                               const T *__restrict__ x, T *__restrict__ y, int lg) {
    const int64_t t = (int64_t)xcd_remap(blockIdx.x, gridDim.x) * 64 + threadIdx.x, i = t >> lg;
    if (i >= g.P) return;             // whole groups of lanes leave together
    const int64_t k = bundle ? bundle[i] : i;
    const int4 rec = walk[k];
    // this lane's steps of the walk: from j0, n of them
    const int part = (int)t & ((1 << lg) - 1);
    const int steps = max(max(abs(rec.y >> 16), abs((int)(int16_t)rec.z)), abs(rec.z >> 16)) + 1;
    const int j0 = steps * part >> lg, n = (steps * (part + 1) >> lg) - j0;
    BresWalk w(rec, j0, g.rvy, 1, g.rvx * g.rvy);
    w.off = (w.z * g.rvx + w.x) * g.rvy + w.y;
    const AccT wt = (AccT)(T)g.scale;
    AccT acc = 0;
    for (int j = 0; j < n; j += 8) {
        T v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            v[u] = x[w.off];
            if (j + u + 1 < n) w.next();   // stays at the last voxel
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (j + u < n) acc += (AccT)v[u] * wt;
    }
    acc = lane_sum(acc, 1 << lg);
    if (part == 0) y[k] = (T)acc;
}

// N of a Siddon operator likewise: sid_walk's steps with eight gathers at a
// time (77 x 101 x 90 voxels, 90,150 rays: 73 -> 32 us, of which the vector
// instructions take 24).  The Siddon operator
// is the FP32 traversal: FP64 products accumulate its weights in FP64 (the
// same matrix in both precisions).
template <typename T, typename AccT>
__global__ __launch_bounds__(64) void k_sid_N(GeoView g, const int32_t *__restrict__ bundle,
                                              const T *__restrict__ x, T *__restrict__ y, int lg) {
#pragma clang fp contract(off)
    const int64_t t = (int64_t)xcd_remap(blockIdx.x, gridDim.x) * 64 + threadIdx.x, i = t >> lg;
    if (i >= g.P) return;             // whole groups of lanes leave together
    const int part = (int)t & ((1 << lg) - 1);
    const int64_t k = bundle ? bundle[i] : i;
    float p0[3], p1[3];
    const int N[3] = {g.rvx, g.rvy, g.rvz};
    const int64_t stride[3] = {g.rvy, 1, (int64_t)g.rvx * g.rvy};
    ray_ends<float>(g, k, p0, p1);
    SidRay<float> s;
    sid_setup(s, p0, p1, g.org, g.h, N);
    AccT acc = 0;
    if (s.hit) {
        // This lane's part of the traversal, event to event: bound j of
        // 1 << lg is the last plane crossing at or before j equal shares.  The
        // entries of the parts are the whole walk's (its state after an event
        // depends on the event's parameter alone).
        auto share = [&](int j) {
            const float p = s.amin + (s.amax - s.amin) * ((float)j / (float)(1 << lg));
            return j == 0 || !(p > s.amin) ? s.amin : (j == 1 << lg || !(p < s.amax) ? s.amax : p);
        };
        auto event = [&](float p) {
            if (!(p > s.amin) || !(p < s.amax)) return p;
            float e = s.amin;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                if (s.st[a] == 0) continue;
                const float before = sid_plane(s, a, sid_next_plane(s, a, p) - s.st[a]);
                e = before > e && before <= p ? before : e;
            }
            return e;
        };
        const float ts = event(share(part)), te = event(share(part + 1));
        // next plane (as a float) and its parameter per axis; a plane beyond
        // the grid lies at or beyond amax, so it is never taken
        float kf[3], tk[3], st[3], tcur = ts;
        int64_t step[3], off = 0;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const bool par = s.st[a] == 0;
            const int kn = par ? 0 : sid_next_plane(s, a, ts);
            const int c = par ? s.cfix[a] : (s.st[a] > 0 ? kn - 1 : kn);
            kf[a] = (float)kn;
            st[a] = (float)s.st[a];
            tk[a] = par ? INFINITY : sid_fma(kf[a], s.A[a], s.B[a]);
            step[a] = s.st[a] * stride[a];
            off += c * stride[a];
        }
        bool on = ts < te;
        for (int left = N[0] + N[1] + N[2] + 4; on && left > 0; left -= 8) {
            float w[8];
            T v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                float tnext = te;
#pragma unroll
                for (int a = 0; a < 3; ++a) tnext = tk[a] < tnext ? tk[a] : tnext;
                w[u] = on ? (tnext - tcur) * s.L : 0.f;
                v[u] = x[off];
                on = on && tnext < te;
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    const bool m = on && tk[a] == tnext;
                    kf[a] += m ? st[a] : 0.f;
                    off += m ? step[a] : 0;
                    tk[a] = m ? sid_fma(kf[a], s.A[a], s.B[a]) : tk[a];
                }
                tcur = on ? tnext : tcur;
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (w[u] > 0) acc = fma((AccT)w[u], (AccT)v[u], acc);
        }
    }
    acc = lane_sum(acc, 1 << lg);
    if (part == 0) y[k] = (T)acc;
}

// T from the rays' parts inside boxes: a workgroup adds the parts of one work
// item into the box in LDS, then writes the box (a box with several items:
// adds it to a cleared y, whole lines at a time).  The sums are FP64 for FP32
// vectors too: an LDS FP64 add serves a wavefront in 22 clocks, an FP32 add
// in 196 (measured, random addresses), which at first bound the kernel: 134
// us at 128^3 with 262,144 Bresenham rays against 44 us now, of which LDS is
// busy 24 and vector issue 21 (1025 us with one memory atomic per entry).
// Parts of equal length are neighbours in the list, so the lanes of a wavefront
// end together.
template <bool SID, typename T>
__global__ __launch_bounds__(kBoxThreads) void k_box_T(GeoView g, int nby, int nbx,
                                                       const int4 *__restrict__ items,
                                                       const uint2 *__restrict__ seg,
                                                       const int4 *__restrict__ walk,
                                                       const float *__restrict__ rec,
                                                       const T *__restrict__ x,
                                                       T *__restrict__ y) {
    constexpr int NV = kRayBoxY * kRayBoxXZ * kRayBoxXZ, NT = kBoxThreads;
    __shared__ double box[NV];
    const int4 it = items[blockIdx.x];
    const int t = threadIdx.x;
    DynPan P = {};
    P.by = it.x % nby * kRayBoxY;
    P.bx = it.x / nby % nbx * kRayBoxXZ;
    P.bz = it.x / nby / nbx * kRayBoxXZ;
    P.bs = kRayBoxXZ;
    P.ey = kRayBoxY;
    P.ez = kRayBoxXZ;
    for (int i = t; i < NV; i += NT) box[i] = 0;
    __syncthreads();
    // a part needs two loads in turn, its segment and then its ray's record
    // and value: segments are requested two parts ahead, records one
    struct Part {
        uint2 sg;
        T xr;
        int4 w;            // Bresenham
        float4 ra, rb;     // Siddon
        float amax;
    };
    auto segment = [&](int k) { return seg[min(k, it.z - 1)]; };
    auto fetch = [&](uint2 sg) {
        Part p = {};
        p.sg = sg;
        p.xr = x[sg.x];
        if constexpr (SID) {
            const float4 *q = reinterpret_cast<const float4 *>(rec + 12 * (int64_t)sg.x);
            p.ra = q[0];
            p.rb = q[1];
            p.amax = q[2].x;
        } else {
            p.w = walk[sg.x];
        }
        return p;
    };
    int k = it.y + t;
    if (k < it.z) {
        Part cur = fetch(segment(k));
        uint2 ahead = segment(k + NT);
        for (; k < it.z; k += NT) {
            const Part nxt = fetch(ahead);
            ahead = segment(k + 2 * NT);
            if (cur.xr != 0) {
                if constexpr (SID) {
                    dyn_seg_walk(DynSeg{cur.ra, cur.rb, cur.amax, (int)cur.sg.y}, P,
                                 [&](int i, float w, bool on) {
                                     if (on) atomicAdd(&box[i], (double)((T)w * cur.xr));
                                 });
                } else {
                    const double v = (double)(cur.xr * (T)g.scale);
                    BresWalk w(cur.w, cur.sg.y & 0xffff, kRayBoxY, 1, kRayBoxY * kRayBoxXZ);
                    w.off = (w.y - P.by) + kRayBoxY * ((w.x - P.bx) + kRayBoxXZ * (w.z - P.bz));
                    for (int j = cur.sg.y >> 16; j > 0; --j) {
                        atomicAdd(&box[w.off & (NV - 1)], v);
                        w.next();
                    }
                }
            }
            cur = nxt;
        }
    }
    __syncthreads();
    for (int i = t; i < NV; i += NT) {
        const int yy = P.by + (i & (kRayBoxY - 1)), xx = P.bx + i / kRayBoxY % kRayBoxXZ,
                  zz = P.bz + i / (kRayBoxY * kRayBoxXZ);
        if (yy >= g.rvy || xx >= g.rvx || zz >= g.rvz) continue;
        const int64_t o = ((int64_t)zz * g.rvx + xx) * g.rvy + yy;
        if (it.w) atomicAdd(&y[o], (T)box[i]);
        else y[o] = (T)box[i];
    }
}

// Bresenham with transducers outside the grid (coordinates clamped)
template <typename T, typename AccT>
__global__ __launch_bounds__(256) void k_clamped_N(GeoView g, const T *__restrict__ x,
                                                   T *__restrict__ y) {
    int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= g.P) return;
    AccT acc = 0;
    int e = g.path[2 * k], r = g.path[2 * k + 1];
    T w = (T)g.scale;
    bresenham_walk(g.ec[3 * e], g.ec[3 * e + 1], g.ec[3 * e + 2], g.rc[3 * r], g.rc[3 * r + 1],
                   g.rc[3 * r + 2], g.rvx, g.rvy, g.rvz,
                   [&](int64_t v) { acc += (AccT)x[v] * (AccT)w; });
    y[k] = (T)acc;
}

// T per ray: FP32 (FP64) hardware atomics on y
template <typename T>
__global__ __launch_bounds__(256) void k_dyn_T(GeoView g, int siddon, const T *__restrict__ x,
                                               T *__restrict__ y) {
    int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= g.P) return;
    const T xr = x[k];
    if (xr == 0) return;
    if (siddon) {
        float p0[3], p1[3];
        int N[3] = {g.rvx, g.rvy, g.rvz};
        ray_ends<float>(g, k, p0, p1);
        siddon_walk<float>(p0, p1, g.org, g.h, N, g.rvy,
                           [&](int64_t v, float w) { atomicAdd(&y[v], (T)w * xr); });
    } else {
        int e = g.path[2 * k], r = g.path[2 * k + 1];
        const T v0 = xr * (T)g.scale;
        bresenham_walk(g.ec[3 * e], g.ec[3 * e + 1], g.ec[3 * e + 2], g.rc[3 * r], g.rc[3 * r + 1],
                       g.rc[3 * r + 2], g.rvx, g.rvy, g.rvz, [&](int64_t v) { atomicAdd(&y[v], v0); });
    }
}

template <typename T>
__global__ void k_clear(int64_t n, T *y) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) y[i] = 0;
}

static int boxes_along(int n, int edge) { return (n + edge - 1) / edge; }

template <typename T, typename AccT>
static void dyn_apply(tv3_op *op, bool trans, const T *x, T *y, hipStream_t s) {
    const DynGeom &G = op->geo;
    const GeoView g = view(G);
    const int sid = G.mode == TV3_WEIGHT_SIDDON;
    const unsigned rays256 = (unsigned)((g.P + 255) / 256);
    if (!trans) {
        // up to eight lanes share a ray, until the chip has 16 wavefronts a CU
        // (4,096 at 256 CUs).  us, one lane a ray -> this: Siddon 57 x 71 x 50,
        // 9,408 rays 18.6 -> 13.2; 77 x 101 x 90, 90,150 33.6 -> 31.9; 121 x 101
        // x 97, 147,456 55 -> 50; Bresenham 50^3, 9,408 8.7 -> 6.2; 64^3, 65,536
        // 11.1 -> 10.2; twice as many lanes 36 and 53, 128^3 76 -> 83
        int lg = 0;
        while (lg < 3 && (g.P << lg) < (int64_t)op->ctx->num_cus * 16 * 64) ++lg;
        const unsigned waves = (unsigned)(((g.P << lg) + 63) / 64);
        if (sid)
            hipLaunchKernelGGL((k_sid_N<T, AccT>), dim3(waves), dim3(64), 0, s, g, G.bundle.p, x, y,
                               lg);
        else if (G.inside)
            hipLaunchKernelGGL((k_bres_N<T, AccT>), dim3(waves), dim3(64), 0, s, g, G.bundle.p,
                               G.walk.p, x, y, lg);
        else
            hipLaunchKernelGGL((k_clamped_N<T, AccT>), dim3(rays256), dim3(256), 0, s, g, x, y);
    } else {
        if (G.boxes.nitem == 0 || G.boxes.split)
            hipLaunchKernelGGL(k_clear<T>, dim3((unsigned)((op->n + 255) / 256)), dim3(256), 0, s,
                               op->n, y);
        const dim3 items((unsigned)G.boxes.nitem);
        const int nby = boxes_along(g.rvy, kRayBoxY), nbx = boxes_along(g.rvx, kRayBoxXZ);
        if (G.boxes.nitem && sid)
            hipLaunchKernelGGL((k_box_T<true, T>), items, dim3(kBoxThreads), 0, s, g, nby, nbx,
                               G.boxes.item.p, G.boxes.seg.p, G.walk.p, G.rec.p, x, y);
        else if (G.boxes.nitem)
            hipLaunchKernelGGL((k_box_T<false, T>), items, dim3(kBoxThreads), 0, s, g, nby, nbx,
                               G.boxes.item.p, G.boxes.seg.p, G.walk.p, G.rec.p, x, y);
        else
            hipLaunchKernelGGL((k_dyn_T<T>), dim3(rays256), dim3(256), 0, s, g, sid, x, y);
    }
    TV3_HIP(hipGetLastError());
}

void dynamic_apply(tv3_op *op, bool trans, const float *x, float *y, hipStream_t s, bool acc64) {
    // a Siddon operator with tile products: deterministic, no atomics
    if (op->kind == OpKind::DYNAMIC && dyn_tile_apply(op, trans, x, y, s)) return;
    acc64 ? dyn_apply<float, double>(op, trans, x, y, s) : dyn_apply<float, float>(op, trans, x, y, s);
}
void dynamic_apply(tv3_op *op, bool trans, const double *x, double *y, hipStream_t s, bool) {
    dyn_apply<double, double>(op, trans, x, y, s);
}

// ------------------------------------------------------------- ray boxes
// Per ray: the walk's record (Bresenham) or the traversal's (Siddon).
__global__ __launch_bounds__(256) void k_ray_records(GeoView g, int siddon, int4 *walk,
                                                     float *rec) {
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= g.P) return;
    if (siddon) {
        float p0[3], p1[3];
        const int N[3] = {g.rvx, g.rvy, g.rvz};
        ray_ends<float>(g, k, p0, p1);
        SidRay<float> s;
        sid_setup(s, p0, p1, g.org, g.h, N);
        float4 *o = reinterpret_cast<float4 *>(rec + 12 * k);
        o[0] = make_float4(s.A[0], s.A[1], s.A[2], s.L);
        o[1] = make_float4(s.B[0], s.B[1], s.B[2], s.amin);
        o[2] = make_float4(s.amax, 0.f, 0.f, 0.f);
    } else {
        const int32_t *a = g.ec + 3 * (int64_t)g.path[2 * k], *b = g.rc + 3 * (int64_t)g.path[2 * k + 1];
        auto two = [](int lo, int hi) { return (int)((unsigned)(lo & 0xffff) | (unsigned)hi << 16); };
        walk[k] = make_int4(two(a[0], a[1]), two(a[2], b[0] - a[0]), two(b[1] - a[1], b[2] - a[2]),
                            0);
    }
}

// Every ray's walk cut at box faces (a box is convex: one part per ray and
// box).  FILL = false: counts the parts; FILL = true: cnt holds the next free
// segment.  A box has a counter for each of kLenClasses lengths, longest
// first (Siddon, whose parts are longer, in steps of two).
template <bool FILL>
__global__ __launch_bounds__(64) void k_box_parts(GeoView g, int siddon,
                                                  const int32_t *__restrict__ bundle, int nby,
                                                  int nbx, int32_t *cnt, uint2 *seg) {
    const int64_t i = (int64_t)blockIdx.x * 64 + threadIdx.x;
    if (i >= g.P) return;
    const int64_t k = bundle ? bundle[i] : i;
    int cur = -1, j = 0;
    unsigned first = 0;
    auto close = [&]() {
        if (cur < 0) return;
        const int len = siddon ? j >> 1 : j - (int)first;
        const int cls = max(kLenClasses - 1 - len, 0);
        const int at = atomicAdd(&cnt[(int64_t)cur * kLenClasses + cls], 1);
        if (FILL)
            seg[at] = make_uint2((unsigned)k, siddon ? first : first | (unsigned)len << 16);
    };
    auto visit = [&](int x, int y, int z) {
        const int b = (z / kRayBoxXZ * nbx + x / kRayBoxXZ) * nby + y / kRayBoxY;
        if (b != cur) {
            close();
            cur = b;
            if (siddon) {
                first = (unsigned)(x % kRayBoxXZ | y % kRayBoxY << 4 | z % kRayBoxXZ << 8);
                j = 0;
            } else {
                first = (unsigned)j;
            }
        }
        ++j;
    };
    if (siddon) {
        float p0[3], p1[3];
        const int N[3] = {g.rvx, g.rvy, g.rvz};
        ray_ends<float>(g, k, p0, p1);
        SidRay<float> s;
        sid_setup(s, p0, p1, g.org, g.h, N);
        if (s.hit)
            sid_walk(s, s.amin, s.amax, [&](int x, int y, int z, float) { visit(x, y, z); });
    } else {
        const int32_t *a = g.ec + 3 * (int64_t)g.path[2 * k], *b = g.rc + 3 * (int64_t)g.path[2 * k + 1];
        bresenham_steps(a[0], a[1], a[2], b[0], b[1], b[2], visit);
    }
    close();
}

// the boxes' segments and work items
static void build_ray_boxes(tv3_ctx *ctx, DynGeom &G) {
    hipStream_t s = ctx->stream;
    const GeoView g = view(G);
    const int sid = G.mode == TV3_WEIGHT_SIDDON;
    const unsigned rays64 = (unsigned)((g.P + 63) / 64);
    const int nby = boxes_along(g.rvy, kRayBoxY), nbx = boxes_along(g.rvx, kRayBoxXZ);
    const int64_t nbox = (int64_t)nby * nbx * boxes_along(g.rvz, kRayBoxXZ);
    const int64_t ncnt = nbox * kLenClasses;
    DevBuf<int32_t> cnt(ncnt), ptr(ncnt + 1);
    TV3_HIP(hipMemsetAsync(cnt.p, 0, cnt.bytes(), s));
    hipLaunchKernelGGL(k_box_parts<false>, dim3(rays64), dim3(64), 0, s, g, sid, G.bundle.p, nby,
                       nbx, cnt.p, (uint2 *)nullptr);
    const int64_t nseg = exclusive_scan_i32(ctx, cnt.p, ptr.p, ncnt);
    G.boxes.seg.alloc(nseg > 0 ? nseg : 1);
    TV3_HIP(hipMemcpyAsync(cnt.p, ptr.p, sizeof(int32_t) * ncnt, hipMemcpyDeviceToDevice, s));
    hipLaunchKernelGGL(k_box_parts<true>, dim3(rays64), dim3(64), 0, s, g, sid, G.bundle.p, nby,
                       nbx, cnt.p, G.boxes.seg.p);
    std::vector<int32_t> q(ncnt + 1), p(nbox + 1);
    TV3_HIP(hipMemcpyAsync(q.data(), ptr.p, sizeof(int32_t) * (ncnt + 1), hipMemcpyDeviceToHost, s));
    TV3_HIP(hipStreamSynchronize(s));
    for (int64_t b = 0; b <= nbox; ++b) p[b] = q[b * kLenClasses];
    std::vector<int4> items;
    for (int64_t b = 0; b < nbox; ++b) {
        const int32_t c = p[b + 1] - p[b], k = std::max(1, (c + kBoxSegs - 1) / kBoxSegs);
        for (int32_t i = 0; i < k; ++i)
            items.push_back(int4{(int)b, (int)(p[b] + (int64_t)c * i / k),
                                 (int)(p[b] + (int64_t)c * (i + 1) / k), k > 1});
        G.boxes.split = G.boxes.split || k > 1;
    }
    std::stable_sort(items.begin(), items.end(),
                     [](const int4 &a, const int4 &b) { return a.z - a.y > b.z - b.y; });
    G.boxes.item.alloc(items.size());
    TV3_HIP(hipMemcpyAsync(G.boxes.item.p, items.data(), sizeof(int4) * items.size(),
                           hipMemcpyHostToDevice, s));
    TV3_HIP(hipStreamSynchronize(s));
    G.boxes.nitem = (int64_t)items.size();
}

void dynamic_prepare(tv3_op *op, bool boxes) {
    DynGeom &G = op->geo;
    tv3_ctx *ctx = op->ctx;
    hipStream_t s = ctx->stream;
    const int sid = G.mode == TV3_WEIGHT_SIDDON;
    // 8 x 8 transducers: the lanes of one wavefront
    const std::vector<int32_t> bundle = ray_bundles(G, 8);
    if (!bundle.empty()) {
        G.bundle.alloc(bundle.size());
        TV3_HIP(hipMemcpyAsync(G.bundle.p, bundle.data(), sizeof(int32_t) * bundle.size(),
                               hipMemcpyHostToDevice, s));
    }
    if (!sid) {
        // epos_h / rpos_h hold the voxel coordinates
        const int lim[3] = {G.rv_x, G.rv_y, G.rv_z};
        G.inside = std::max({G.rv_x, G.rv_y, G.rv_z}) < 32768 && op->n < (int64_t(1) << 31);
        for (const std::vector<float> *c : {&G.epos_h, &G.rpos_h})
            for (size_t k = 0; k < c->size(); ++k)
                G.inside = G.inside && (*c)[k] >= 0 && (*c)[k] < lim[k % 3];
    }
    const GeoView g = view(G);
    const unsigned rays256 = (unsigned)((g.P + 255) / 256);
    if (!sid && G.inside) G.walk.alloc(g.P);
    if (sid && boxes) G.rec.alloc(12 * g.P);
    if (G.walk.p || G.rec.p)
        hipLaunchKernelGGL(k_ray_records, dim3(rays256), dim3(256), 0, s, g, sid, G.walk.p,
                           G.rec.p);
    // at most one part per ray and box face crossed: their count must fit 32 bits
    const int64_t parts = boxes_along(g.rvy, kRayBoxY) + boxes_along(g.rvx, kRayBoxXZ) +
                          (int64_t)boxes_along(g.rvz, kRayBoxXZ);
    if (boxes && (sid || G.inside) && op->n < (int64_t(1) << 31) && g.P * parts < (int64_t(1) << 31)) {
        try {
            build_ray_boxes(ctx, G);
        } catch (const tv3_error &e) {
            if (e.status != TV3_E_NOMEM) throw;
            G.boxes = RayBoxes();      // the per-ray kernel needs no memory
        }
    }
    TV3_HIP(hipGetLastError());
    TV3_HIP(hipStreamSynchronize(s));
}

// ------------------------------------------------------------- materialize
// Pass 1: each ray walks once into a fixed-capacity slot of a scratch buffer
// (capacity = the longest possible walk) and records its count; the counts
// are scanned into the row pointer; pass 2 compacts the slots into the CSR,
// converting the weights to the storage type.
__global__ __launch_bounds__(256) void k_walk_to_slots(GeoView g, int siddon, int cap,
                                                       int32_t *cnt, int32_t *scol,
                                                       float *sval) {
    int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= g.P) return;
    int c = 0;
    int32_t *oc = scol + k * cap;
    float *ov = sval + k * cap;
    if (siddon) {
        float p0[3], p1[3];
        int N[3] = {g.rvx, g.rvy, g.rvz};
        ray_ends<float>(g, k, p0, p1);
        siddon_walk<float>(p0, p1, g.org, g.h, N, g.rvy, [&](int64_t v, float w) {
            if (c < cap) { oc[c] = (int32_t)v; ov[c] = w; }
            ++c;
        });
    } else {
        int e = g.path[2 * k], r = g.path[2 * k + 1];
        bresenham_walk(g.ec[3 * e], g.ec[3 * e + 1], g.ec[3 * e + 2], g.rc[3 * r], g.rc[3 * r + 1],
                       g.rc[3 * r + 2], g.rvx, g.rvy, g.rvz, [&](int64_t v) {
                           if (c < cap) { oc[c] = (int32_t)v; ov[c] = g.scale; }
                           ++c;
                       });
    }
    cnt[k] = c < cap ? c : cap;
}

template <typename V> __device__ __forceinline__ V cvt(float w);
template <> __device__ __forceinline__ float cvt<float>(float w) { return w; }
template <> __device__ __forceinline__ __half cvt<__half>(float w) { return __float2half(w); }
template <> __device__ __forceinline__ __hip_bfloat16 cvt<__hip_bfloat16>(float w) {
    return __float2bfloat16(w);
}

template <typename V>
__global__ __launch_bounds__(256) void k_compact(int64_t P, int cap, const int32_t *rowptr,
                                                 const int32_t *scol, const float *sval,
                                                 int32_t *col, V *val) {
    int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= P) return;
    int b = rowptr[k], e = rowptr[k + 1];
    for (int j = 0; j < e - b; ++j) {
        col[b + j] = scol[k * cap + j];
        val[b + j] = cvt<V>(sval[k * cap + j]);
    }
}

void dynamic_materialize(tv3_op *op, tv3_dtype vt, SparseRows &A) {
    TV3_REQUIRE(vt == TV3_F32 || vt == TV3_F16 || vt == TV3_BF16, TV3_E_FORMAT,
                "materialized weights must be F32, F16 or BF16");
    tv3_ctx *ctx = op->ctx;
    hipStream_t s = ctx->stream;
    GeoView g = view(op->geo);
    int cap = g.rvx + g.rvy + g.rvz + 4;
    if (op->geo.mode == TV3_WEIGHT_BRESENHAM) cap = op->geo.max_walk;
    A.rows = g.P;
    A.cols = op->n;
    A.vtype = vt;
    A.ptr.alloc(g.P + 1);
    // process rays in chunks so the slot buffer stays bounded (<= ~1 GiB)
    int64_t chunk = (int64_t)((1ll << 30) / (8ll * cap));
    if (chunk < 1) chunk = 1;
    if (chunk > g.P) chunk = g.P > 0 ? g.P : 1;
    DevBuf<int32_t> cnt(g.P > 0 ? g.P : 1), scol(chunk * cap);
    DevBuf<float> sval(chunk * cap);
    int sid = op->geo.mode == TV3_WEIGHT_SIDDON;
    // count pass over all chunks (walk into slots, keep only counts)
    for (int64_t c0 = 0; c0 < g.P; c0 += chunk) {
        GeoView gc = g;
        int64_t cn = g.P - c0 < chunk ? g.P - c0 : chunk;
        gc.P = cn;
        gc.path = g.path + 2 * c0;
        hipLaunchKernelGGL(k_walk_to_slots, dim3((unsigned)((cn + 255) / 256)), dim3(256), 0, s, gc,
                           sid, cap, cnt.p + c0, scol.p, sval.p);
    }
    TV3_HIP(hipGetLastError());
    A.nnz = exclusive_scan_i32(ctx, cnt.p, A.ptr.p, g.P);
    A.ind.alloc(A.nnz > 0 ? A.nnz : 1);
    A.val.alloc((A.nnz > 0 ? A.nnz : 1) * dtype_size(vt));
    for (int64_t c0 = 0; c0 < g.P; c0 += chunk) {
        GeoView gc = g;
        int64_t cn = g.P - c0 < chunk ? g.P - c0 : chunk;
        gc.P = cn;
        gc.path = g.path + 2 * c0;
        unsigned bl = (unsigned)((cn + 255) / 256);
        hipLaunchKernelGGL(k_walk_to_slots, dim3(bl), dim3(256), 0, s, gc, sid, cap, cnt.p + c0,
                           scol.p, sval.p);
        const int32_t *rp = A.ptr.p + c0;
        switch (vt) {
        case TV3_F32:
            hipLaunchKernelGGL(k_compact<float>, dim3(bl), dim3(256), 0, s, cn, cap, rp, scol.p,
                               sval.p, A.ind.p, reinterpret_cast<float *>(A.val.p));
            break;
        case TV3_F16:
            hipLaunchKernelGGL(k_compact<__half>, dim3(bl), dim3(256), 0, s, cn, cap, rp, scol.p,
                               sval.p, A.ind.p, reinterpret_cast<__half *>(A.val.p));
            break;
        default:
            hipLaunchKernelGGL(k_compact<__hip_bfloat16>, dim3(bl), dim3(256), 0, s, cn, cap, rp,
                               scol.p, sval.p, A.ind.p,
                               reinterpret_cast<__hip_bfloat16 *>(A.val.p));
            break;
        }
    }
    TV3_HIP(hipGetLastError());
    TV3_HIP(hipStreamSynchronize(s));
    A.lanes = default_lanes(A.rows, A.nnz);
    build_default_blocks(ctx, A, true);
}

}  // namespace tv3
