// vec.hpp -- declarations of the plain-path vector kernels and the shared
// block-reduction helper.
#pragma once

#include <array>

#include "lanes.hpp"
#include "tv3_internal.hpp"

namespace tv3 {

// Sum K per-thread doubles over a workgroup of NW wavefronts (4: 256
// threads, 8: 512) -- wavefront sums (wave_sum), then the wavefront totals
// in a fixed order; thread 0 stores partials[k*nblk + slot].  Every thread of
// the workgroup calls it.
template <int K, int NW = 4>
__device__ __forceinline__ void block_sum_store_at(double (&acc)[K], double *partials, int nblk,
                                                   int slot) {
    __shared__ double sh[K][NW];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const double v = wave_sum(acc[k]);
        if (lane == 0) sh[k][wave] = v;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            double v = (sh[k][0] + sh[k][1]) + (sh[k][2] + sh[k][3]);
            if (NW == 8) v += (sh[k][4] + sh[k][5]) + (sh[k][6] + sh[k][7]);
            partials[(int64_t)k * nblk + slot] = v;
        }
    }
}

// The same at the workgroup's own slot (blockIdx.x).
template <int K, int NW = 4>
__device__ __forceinline__ void block_sum_store(double (&acc)[K], double *partials, int nblk) {
    block_sum_store_at<K, NW>(acc, partials, nblk, (int)blockIdx.x);
}

// Sums over items, queued as kernels that leave FP64 block partials (at most
// kSumBlocks per sum), and fetched together: one more kernel adds the
// partials and writes value and ticket of each sum to pinned host memory,
// where the host watches for them.  20 iterations of the plain solver at 64^3
// voxels take 1,760 us, against 2,090 with the partials in pinned memory, a
// stream synchronisation, and up to 9,700 additions on the host in each.
// drain: wait for the stream instead, for results that a caller goes on to
// use outside it.
constexpr int kSumBlocks = 1024, kSumMax = 16;
struct Sums {
    tv3_ctx *ctx;
    hipStream_t s;
    size_t used = 0;
    int count = 0;
    struct Sum {
        int first, stride, blocks;
    } sum[kSumMax] = {};
    double value[kSumMax] = {};
    const double *fetch(bool drain = false);     // the sums in the order queued
};

// the volume-sized fields the plain loop's fused steps share
template <typename T> struct PlainFields {
    const int32_t *dims;
    int64_t n;
    const T *Ux, *Uy, *Uz;       // D U
    T *Wx, *Wy, *Wz;
    const T *sx, *sy, *sz;       // sigma
    T *g2;                       // D^T (D U - W)
};

// V = U - tau d (clamped at 0 with nonneg) and its differences D V
template <typename T>
void descend_step(const int32_t dims[3], double tau, bool nonneg, const T *U, const T *d, T *V,
                  T *Vx, T *Vy, T *Vz, hipStream_t s);
// |D d|^2 along x, y, z and |d|^2
template <typename T> void queue_step(Sums &S, const int32_t dims[3], const T *d);
template <typename T> void queue_dot(Sums &S, int64_t n, const T *a, const T *b);
// lam2, lam4, g2 = D^T (DU - W), g = (A^T Au) - Atb (g NULL: not formed), and
// lam3, lam5
template <typename T>
void queue_gradient(Sums &S, const PlainFields<T> &f, T *g, const T *Atb, int64_t m, const T *Au,
                    const T *b, const T *delta);
// the same and queue_shrink of the next W's fields, which neither reads what
// the other writes, in one launch
template <typename T>
void queue_trial(Sums &S, const PlainFields<T> &f, T *g, const T *Atb, int64_t m, const T *Au,
                 const T *b, const T *delta, const PlainFields<T> &next, int iso, double beta);
// lam2, lam4
template <typename T> void queue_lam24(Sums &S, const PlainFields<T> &f);
// lam3, lam5
template <typename T>
void queue_lam35(Sums &S, int64_t m, const T *Au, const T *b, const T *delta);
// W; lam1
template <typename T> void queue_shrink(Sums &S, const PlainFields<T> &f, int iso, double beta);
// g2, d; lam2, lam4, |d|^2, |U - Up|^2, |Up|^2, <U - Up, change of the gradient>
template <typename T>
void queue_update(Sums &S, const PlainFields<T> &f, const T *g, const T *gp, const T *g2p,
                  const T *dts, const T *U, const T *Up, double mdb, T *d);

template <typename T> void axpy3(int64_t n, T *z, double a, const T *x, const T *y, hipStream_t s);
template <typename T>
void grad(int64_t n, T *d, double a, const T *g, const T *g2, const T *dts, hipStream_t s);
template <typename T> void scale(int64_t n, T *y, double a, const T *x, hipStream_t s);
template <typename T> void divide(int64_t n, T *y, double a, const T *x, hipStream_t s);
template <typename T>
double mlp_sigma(tv3_ctx *ctx, int64_t n, const T *Ux, const T *Uy, const T *Uz, const T *Wx,
                 const T *Wy, const T *Wz, double beta, T *sx, T *sy, T *sz, hipStream_t s);
template <typename T>
double mlp_delta(tv3_ctx *ctx, int64_t m, const T *Au, const T *b, double mu, T *delta,
                 hipStream_t s);
template <typename T>
std::array<double, 2> diff_norm(tv3_ctx *ctx, int64_t n, const T *a, const T *b, hipStream_t s);

}  // namespace tv3
