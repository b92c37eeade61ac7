// dense.hip -- column-major dense products (gemv N and T), the semantics of
// dense_mm / mat_vec_mul (3d/mat_vec_mul_dense.h:25-73: gemv with alpha = 1,
// beta = 0, leading dimension lda).
//
// Both are bound by reading A once, so both load it 16 bytes a lane (W = 16 /
// sizeof(V) entries of one column; a wavefront load is 1 KB of one column).
// Measured against one entry a lane and load: 8192 x 16384 BF16, N 108 + 36
// (partial sums) -> 40 + 5 us, T 107 -> 50 us (6.7 and 5.4 TB/s of a matrix
// partly in the memory-side cache); 1638 x 4096 FP32, N 20 + 17 -> 6.6 + 2.6
// us, T 10.3 -> 6.9 us.
// Columns start at any multiple of the element size (lda and the caller's
// matrix decide), so the loads are declared with the element's alignment.
//
// N (y = A x): a wavefront owns 64 W rows and walks columns, eight loads in
// flight; the four wavefronts of a workgroup walk neighbouring column runs of
// the same rows and add up in LDS; gridDim.y column slabs fill the chip and
// their partial sums are added by a second kernel.  Fixed orders, no atomics.
// T (y = A^T x): a wavefront owns C columns and walks their rows, so that W
// values of x in registers serve C loads of A (with one column, x is 2 bytes
// of L1 traffic per byte of a BF16 matrix and set the pace).
#include <algorithm>
#include <optional>

#include "lanes.hpp"
#include "tv3_internal.hpp"

namespace tv3 {

namespace {

// W consecutive values at any multiple of their own size
template <typename V, int W>
struct __attribute__((packed, aligned(alignof(V)))) Run {
    V v[W];
};

template <typename V, int W>
__device__ __forceinline__ Run<V, W> load_run(const V *p) {
    return *reinterpret_cast<const Run<V, W> *>(p);
}

template <typename AccT, typename V>
__device__ __forceinline__ AccT up(V v) {
    if constexpr (std::is_same<V, __half>::value) return (AccT)__half2float(v);
    else if constexpr (std::is_same<V, __hip_bfloat16>::value) return (AccT)__bfloat162float(v);
    else return (AccT)v;
}

// entries per lane and load: 16 bytes' worth
template <typename V> constexpr int run_of() { return 16 / (int)sizeof(V); }

constexpr int kColsInFlight = 8;

// Rows beyond the last whole run are covered by moving the last lanes' runs
// back to end at row m (m >= W): a row held by two lanes gets the same sum
// twice and both store it.
template <typename V, int W, int KT, typename T, typename AccT>
__global__ __launch_bounds__(256) void k_gemv_n_part(int64_t m, int64_t n, int64_t lda,
                                                     const V *__restrict__ A,
                                                     const T *__restrict__ x, int64_t ldx, int G,
                                                     AccT *__restrict__ part, T *__restrict__ y,
                                                     int64_t ldy, int64_t cols_per) {
    __shared__ AccT sh[3][64 * W];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t i = min(((int64_t)blockIdx.x * 64 + lane) * W, m - W);
    const int64_t s0 = (int64_t)blockIdx.y * cols_per, s1 = min(s0 + cols_per, n);
    const int64_t per = (cols_per + 3) / 4;
    const int64_t j0 = min(s0 + wave * per, s1), j1 = min(j0 + per, s1);
    AccT s[KT][W] = {};
    const V *a = A + i + j0 * lda;
    const T *xk[KT];
#pragma unroll
    for (int k = 0; k < KT; ++k) xk[k] = x + (int64_t)min(k, G - 1) * ldx;
    int64_t j = j0;
    for (; j + kColsInFlight <= j1; j += kColsInFlight, a += kColsInFlight * lda) {
        Run<V, W> r[kColsInFlight];
#pragma unroll
        for (int c = 0; c < kColsInFlight; ++c) r[c] = load_run<V, W>(a + c * lda);
#pragma unroll
        for (int c = 0; c < kColsInFlight; ++c)
#pragma unroll
            for (int k = 0; k < KT; ++k) {
                const AccT xj = (AccT)xk[k][j + c];
#pragma unroll
                for (int e = 0; e < W; ++e) s[k][e] += up<AccT>(r[c].v[e]) * xj;
            }
    }
    for (; j < j1; ++j, a += lda) {
        const Run<V, W> r = load_run<V, W>(a);
#pragma unroll
        for (int k = 0; k < KT; ++k) {
            const AccT xj = (AccT)xk[k][j];
#pragma unroll
            for (int e = 0; e < W; ++e) s[k][e] += up<AccT>(r.v[e]) * xj;
        }
    }
#pragma unroll
    for (int k = 0; k < KT; ++k) {
        if (k > 0) __syncthreads();          // the previous vector's sums have been read
        if (wave > 0) {
#pragma unroll
            for (int e = 0; e < W; ++e) sh[wave - 1][e * 64 + lane] = s[k][e];
        }
        __syncthreads();
        if (wave > 0 || k >= G) continue;
#pragma unroll
        for (int e = 0; e < W; ++e) {
            const AccT t = (s[k][e] + sh[0][e * 64 + lane]) +
                           (sh[1][e * 64 + lane] + sh[2][e * 64 + lane]);
            if (gridDim.y == 1) y[k * ldy + i + e] = (T)t;
            else part[((int64_t)k * gridDim.y + blockIdx.y) * m + i + e] = t;
        }
    }
}

// y = sum of the ks slab partials: 64 rows a workgroup, its wavefronts each a
// quarter of the slabs (one thread summing all slabs of a row was a chain of
// up to 128 dependent loads); blockIdx.y is the vector.
template <typename T, typename AccT>
__global__ __launch_bounds__(256) void k_gemv_n_sum(int64_t m, int ks,
                                                    const AccT *__restrict__ part,
                                                    T *__restrict__ y, int64_t ldy) {
    __shared__ AccT sh[3][64];
    part += (int64_t)blockIdx.y * ks * m;
    y += blockIdx.y * ldy;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t i = min((int64_t)blockIdx.x * 64 + lane, m - 1);
    AccT s = 0;
    int k = wave;
    for (; k + 28 < ks; k += 32) {
        AccT v[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) v[c] = part[(int64_t)(k + 4 * c) * m + i];
        s += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    }
    for (; k < ks; k += 4) s += part[(int64_t)k * m + i];
    if (wave > 0) sh[wave - 1][lane] = s;
    __syncthreads();
    if (wave == 0) y[i] = (T)((s + sh[0][lane]) + (sh[1][lane] + sh[2][lane]));
}

template <typename V, int W, int C, int KT, typename T, typename AccT>
__global__ __launch_bounds__(256) void k_gemv_t(int64_t m, int64_t n, int64_t lda,
                                                const V *__restrict__ A,
                                                const T *__restrict__ x, int64_t ldx, int G,
                                                T *__restrict__ y, int64_t ldy) {
    const int lane = threadIdx.x & 63;
    const int64_t j0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * C;
    if (j0 >= n) return;
    const V *col[C];
#pragma unroll
    for (int c = 0; c < C; ++c) col[c] = A + min(j0 + c, n - 1) * lda;
    const T *xk[KT];
#pragma unroll
    for (int k = 0; k < KT; ++k) xk[k] = x + (int64_t)min(k, G - 1) * ldx;
    AccT s[C][KT] = {}, s2[C][KT] = {};
    auto add = [&](const Run<V, W> &r, const Run<T, W> &xv, AccT &sum) {
        AccT p = 0;
#pragma unroll
        for (int e = 0; e < W; ++e) p += up<AccT>(r.v[e]) * (AccT)xv.v[e];
        sum += p;
    };
    const int64_t step = 64 * W, whole = m / step * step;
    int64_t i = (int64_t)lane * W;
    for (; i + step < whole; i += 2 * step) {
        Run<V, W> r[C], r2[C];
        Run<T, W> xv[KT], xv2[KT];
#pragma unroll
        for (int k = 0; k < KT; ++k) {
            xv[k] = load_run<T, W>(xk[k] + i);
            xv2[k] = load_run<T, W>(xk[k] + i + step);
        }
#pragma unroll
        for (int c = 0; c < C; ++c) {
            r[c] = load_run<V, W>(col[c] + i);
            r2[c] = load_run<V, W>(col[c] + i + step);
        }
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int k = 0; k < KT; ++k) {
                add(r[c], xv[k], s[c][k]);
                add(r2[c], xv2[k], s2[c][k]);
            }
    }
    for (; i + W <= m; i += step) {
        Run<T, W> xv[KT];
#pragma unroll
        for (int k = 0; k < KT; ++k) xv[k] = load_run<T, W>(xk[k] + i);
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const Run<V, W> r = load_run<V, W>(col[c] + i);
#pragma unroll
            for (int k = 0; k < KT; ++k) add(r, xv[k], s[c][k]);
        }
    }
    // the rows after the last whole run: one a lane
    const int64_t tail = m / W * W + lane;
    if (tail < m) {
#pragma unroll
        for (int k = 0; k < KT; ++k) {
            const AccT xv = (AccT)xk[k][tail];
#pragma unroll
            for (int c = 0; c < C; ++c) s2[c][k] += up<AccT>(col[c][tail]) * xv;
        }
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int k = 0; k < KT; ++k) {
            const AccT t = lane_sum<64>(s[c][k] + s2[c][k]);
            if (lane == 0 && j0 + c < n && k < G) y[k * ldy + j0 + c] = (T)t;
        }
}

}  // namespace

// Column slabs of A x: enough workgroups for four a CU, as far as the columns
// go; never more than the min(128, ceil(n / 64)) that a workspace of the
// caller's is checked for.
static int64_t most_slabs(int64_t n) {
    const int64_t slabs = std::min<int64_t>(128, (n + 63) / 64), per = (n + slabs - 1) / slabs;
    return (n + per - 1) / per;
}
static int64_t slabs_of(const tv3_op *op, int W) {
    const int64_t tiles = (op->m + 64 * W - 1) / (64 * W), n = op->n;
    const int64_t ks = std::min(most_slabs(n),
                                std::max<int64_t>(1, (4 * op->ctx->num_cus + tiles - 1) / tiles));
    const int64_t per = (n + ks - 1) / ks;
    return (n + per - 1) / per;
}

// G vectors (1 <= G <= KT).  ws: the split-K partials of A x go to this
// workspace of ws_bytes (the allocation-free path, one vector) instead of the
// context's, which grows on demand to what the launch uses.
template <typename V, int W, int KT, typename T, typename AccT>
static void gemv_n(tv3_op *op, int G, const T *x, int64_t ldx, T *y, int64_t ldy, hipStream_t s,
                   void *ws, size_t ws_bytes) {
    const V *A = reinterpret_cast<const V *>(op->dense.p);
    const int64_t m = op->m, n = op->n, lda = op->lda;
    if (ws) {
        const size_t most = sizeof(AccT) * (size_t)most_slabs(n) * (size_t)m;
        TV3_REQUIRE(most <= ws_bytes, TV3_E_UNSUPPORTED,
                    "dense A x needs " + std::to_string(most) + " bytes of partial sums; the "
                    "allocation-free path holds " + std::to_string(ws_bytes));
    }
    const int64_t tiles = (m + 64 * W - 1) / (64 * W);
    const int64_t ks = slabs_of(op, W), cols_per = (n + ks - 1) / ks;
    AccT *part = reinterpret_cast<AccT *>(ws);
    std::optional<StreamScratch::Lease> lease;
    if (!ws && ks > 1) {
        lease.emplace(op->ctx->scratch.take(s, sizeof(AccT) * (size_t)(ks * m) * (size_t)G));
        part = reinterpret_cast<AccT *>(lease->p);
    }
    hipLaunchKernelGGL((k_gemv_n_part<V, W, KT, T, AccT>), dim3((unsigned)tiles, (unsigned)ks),
                       dim3(256), 0, s, m, n, lda, A, x, ldx, G, part, y, ldy, cols_per);
    if (ks > 1)
        hipLaunchKernelGGL((k_gemv_n_sum<T, AccT>), dim3((unsigned)((m + 63) / 64), (unsigned)G),
                           dim3(256), 0, s, m, (int)ks, part, y, ldy);
}

template <typename V, int C, int KT, typename T, typename AccT>
static void gemv_t(tv3_op *op, int G, const T *x, int64_t ldx, T *y, int64_t ldy, hipStream_t s) {
    constexpr int W = run_of<V>();
    hipLaunchKernelGGL((k_gemv_t<V, W, C, KT, T, AccT>),
                       dim3((unsigned)((op->n + 4 * C - 1) / (4 * C))), dim3(256), 0, s, op->m,
                       op->n, op->lda, reinterpret_cast<const V *>(op->dense.p), x, ldx, G, y, ldy);
}

template <typename V, int KT, typename T, typename AccT>
static void gemv(tv3_op *op, bool trans, int G, const T *x, int64_t ldx, T *y, int64_t ldy,
                 hipStream_t s, void *ws = nullptr, size_t ws_bytes = 0) {
    constexpr int W = run_of<V>();
    if (!trans) {
        if (op->m >= W) gemv_n<V, W, KT, T, AccT>(op, G, x, ldx, y, ldy, s, ws, ws_bytes);
        else gemv_n<V, 1, KT, T, AccT>(op, G, x, ldx, y, ldy, s, ws, ws_bytes);
    } else {
        // columns per wavefront: as many as leave eight wavefronts a CU
        const int64_t waves = 8 * (int64_t)op->ctx->num_cus;
        if (op->n >= 4 * waves) gemv_t<V, 4, KT, T, AccT>(op, G, x, ldx, y, ldy, s);
        else if (op->n >= 2 * waves) gemv_t<V, 2, KT, T, AccT>(op, G, x, ldx, y, ldy, s);
        else gemv_t<V, 1, KT, T, AccT>(op, G, x, ldx, y, ldy, s);
    }
    TV3_HIP(hipGetLastError());
}

// one vector
template <typename V, typename T, typename AccT>
static void gemv(tv3_op *op, bool trans, const T *x, T *y, hipStream_t s, void *ws = nullptr,
                 size_t ws_bytes = 0) {
    gemv<V, 1, T, AccT>(op, trans, 1, x, 0, y, 0, s, ws, ws_bytes);
}

// Several vectors, each with its single product's additions in the same
// order (same bits): a reading of A serves up to eight.  2047 x 8190 FP32, 8
// vectors, A X 448 -> 20 us and A^T R 105 -> 18 us (26 four at a time); 64
// vectors 3579 -> 155 and 831 -> 137 us; 4000 x 16001 BF16, 8 vectors, 571 ->
// 34 and 342 -> 47 us (one at a time, before).
template <typename V>
static void gemv_multi(tv3_op *op, bool trans, int nrhs, const float *X, int64_t ldx, float *Y,
                       int64_t ldy, hipStream_t s) {
    for (int j = 0; j < nrhs;) {
        const int left = std::min(nrhs - j, 8);
        const float *x = X + j * ldx;
        float *y = Y + j * ldy;
        if (left == 1) {
            gemv<V, 1, float, float>(op, trans, 1, x, ldx, y, ldy, s);
        } else if (left == 2) {
            gemv<V, 2, float, float>(op, trans, 2, x, ldx, y, ldy, s);
        } else if (left <= 4) {
            gemv<V, 4, float, float>(op, trans, left, x, ldx, y, ldy, s);
        } else {
            gemv<V, 8, float, float>(op, trans, left, x, ldx, y, ldy, s);
        }
        j += left;
    }
}

void dense_gemv_multi(tv3_op *op, bool trans, int nrhs, const float *X, int64_t ldx, float *Y,
                      int64_t ldy, hipStream_t s) {
    switch (op->dtype) {
    case TV3_F32: gemv_multi<float>(op, trans, nrhs, X, ldx, Y, ldy, s); break;
    case TV3_F16: gemv_multi<__half>(op, trans, nrhs, X, ldx, Y, ldy, s); break;
    case TV3_BF16: gemv_multi<__hip_bfloat16>(op, trans, nrhs, X, ldx, Y, ldy, s); break;
    default: throw tv3_error(TV3_E_FORMAT, "FP32 dense products need F32, F16 or BF16 values");
    }
}

void dense_gemv(tv3_op *op, bool trans, const float *x, float *y, hipStream_t s, bool acc64) {
    switch (op->dtype) {
    case TV3_F32:
        acc64 ? gemv<float, float, double>(op, trans, x, y, s) : gemv<float, float, float>(op, trans, x, y, s);
        break;
    case TV3_F16:
        acc64 ? gemv<__half, float, double>(op, trans, x, y, s)
              : gemv<__half, float, float>(op, trans, x, y, s);
        break;
    case TV3_BF16:
        acc64 ? gemv<__hip_bfloat16, float, double>(op, trans, x, y, s)
              : gemv<__hip_bfloat16, float, float>(op, trans, x, y, s);
        break;
    default: throw tv3_error(TV3_E_FORMAT, "FP32 dense products need F32, F16 or BF16 values");
    }
}

void dense_gemv_ws(tv3_op *op, const float *x, float *y, hipStream_t s, void *ws,
                   size_t ws_bytes) {
    switch (op->dtype) {
    case TV3_F32: gemv<float, float, float>(op, false, x, y, s, ws, ws_bytes); break;
    case TV3_F16: gemv<__half, float, float>(op, false, x, y, s, ws, ws_bytes); break;
    case TV3_BF16: gemv<__hip_bfloat16, float, float>(op, false, x, y, s, ws, ws_bytes); break;
    default: throw tv3_error(TV3_E_FORMAT, "FP32 dense products need F32, F16 or BF16 values");
    }
}

void dense_gemv(tv3_op *op, bool trans, const double *x, double *y, hipStream_t s, bool) {
    switch (op->dtype) {
    case TV3_F64: gemv<double, double, double>(op, trans, x, y, s); break;
    case TV3_F32: gemv<float, double, double>(op, trans, x, y, s); break;
    default: throw tv3_error(TV3_E_FORMAT, "FP64 dense products need F64 or F32 values");
    }
}

}  // namespace tv3
