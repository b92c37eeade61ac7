// vec.hip -- vector kernels of the reference-shaped ("plain") TVAL3 loop: the
// operations between two host decisions share kernels, reductions are FP64 block
// partials totalled on the device in a fixed order.  Float and double
// instantiations.
//
// Reference kernels restated (3d/tval3_gpu_3d_kernels.cu): vec_add :75-108,
// D :170-215, D^T :479-510, lam2/lam4 :724-771 (all three components, sigma
// in X,Y,Z order), lam3/lam5 :876-919, BB step :1017-1067, nonneg
// :1176-1188, shrinkage :1249-1300 (plus the isotropic variant).
#include <chrono>

#include "vec.hpp"

namespace tv3 {

// ---------------------------------------------------------------- elementwise
template <typename T>
__global__ void k_axpy3(int64_t n, T *z, T a, const T *x, const T *y) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        z[i] = a * x[i] + y[i];
}

template <typename T>
__global__ void k_grad(int64_t n, T *d, T a, const T *g, const T *g2, const T *dts) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        T v = a * g[i] + g2[i];
        d[i] = v + dts[i];
    }
}

template <typename T>
__global__ void k_scale(int64_t n, T *y, T a, const T *x) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        y[i] = a * x[i];
}

template <typename T>
__global__ void k_div(int64_t n, T *y, T a, const T *x) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        y[i] = x[i] / a;
}

static inline unsigned ew_blocks(int64_t n) {
    int64_t b = (n + 255) / 256;
    if (b > 8192) b = 8192;
    return (unsigned)(b > 0 ? b : 1);
}

template <typename T>
void axpy3(int64_t n, T *z, double a, const T *x, const T *y, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_axpy3<T>, dim3(ew_blocks(n)), dim3(256), 0, s, n, z, (T)a, x, y);
}
template <typename T>
void grad(int64_t n, T *d, double a, const T *g, const T *g2, const T *dts, hipStream_t s) {
    hipLaunchKernelGGL(k_grad<T>, dim3(ew_blocks(n)), dim3(256), 0, s, n, d, (T)a, g, g2, dts);
}
template <typename T>
void divide(int64_t n, T *y, double a, const T *x, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_div<T>, dim3(ew_blocks(n)), dim3(256), 0, s, n, y, (T)a, x);
}
template <typename T>
void scale(int64_t n, T *y, double a, const T *x, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_scale<T>, dim3(ew_blocks(n)), dim3(256), 0, s, n, y, (T)a, x);
}

// ---------------------------------------------------------------- stencils
// thread (tx, ty) of block (bx, by, bz) owns voxel y = bx*64+tx, x = by*4+ty, z = bz
template <typename T>
__global__ __launch_bounds__(256) void k_D(int p, int q, int r, const T *__restrict__ U,
                                           T *__restrict__ Ux, T *__restrict__ Uy,
                                           T *__restrict__ Uz) {
    int y = blockIdx.x * 64 + threadIdx.x, x = blockIdx.y * 4 + threadIdx.y, z = blockIdx.z;
    if (y >= p || x >= q) return;
    int64_t pq = (int64_t)p * q;
    int64_t i = (int64_t)z * pq + (int64_t)x * p + y;
    T t = U[i];
    Uy[i] = (y < p - 1 ? U[i + 1] : U[i - y]) - t;
    Ux[i] = (x < q - 1 ? U[i + p] : U[i - (int64_t)x * p]) - t;
    Uz[i] = (z < r - 1 ? U[i + pq] : U[i - (int64_t)z * pq]) - t;
}

template <typename T>
__global__ __launch_bounds__(256) void k_Dt(int p, int q, int r, const T *__restrict__ X,
                                            const T *__restrict__ Y, const T *__restrict__ Z,
                                            T *__restrict__ res) {
    int y = blockIdx.x * 64 + threadIdx.x, x = blockIdx.y * 4 + threadIdx.y, z = blockIdx.z;
    if (y >= p || x >= q) return;
    int64_t pq = (int64_t)p * q;
    int64_t i = (int64_t)z * pq + (int64_t)x * p + y;
    T yp = (y == 0) ? Y[i + p - 1] : Y[i - 1];
    T xp = (x == 0) ? X[i + (int64_t)(q - 1) * p] : X[i - p];
    T zp = (z == 0) ? Z[i + (int64_t)(r - 1) * pq] : Z[i - pq];
    res[i] = yp - Y[i] + xp - X[i] + zp - Z[i];
}

static inline dim3 st_grid(const int32_t dims[3]) {
    return dim3((unsigned)((dims[0] + 63) / 64), (unsigned)((dims[1] + 3) / 4), (unsigned)dims[2]);
}

template <typename T>
void launch_D(const int32_t dims[3], const T *U, T *Ux, T *Uy, T *Uz, hipStream_t s) {
    hipLaunchKernelGGL(k_D<T>, st_grid(dims), dim3(64, 4), 0, s, dims[0], dims[1], dims[2], U, Ux,
                       Uy, Uz);
}
template <typename T>
void launch_Dt(const int32_t dims[3], const T *X, const T *Y, const T *Z, T *res, hipStream_t s) {
    hipLaunchKernelGGL(k_Dt<T>, st_grid(dims), dim3(64, 4), 0, s, dims[0], dims[1], dims[2], X, Y,
                       Z, res);
}

// ---------------------------------------------------------------- reductions
template <typename T> struct FDot {
    const T *a, *b;
    __device__ void operator()(int64_t i, double *acc) const { acc[0] += (double)a[i] * (double)b[i]; }
};

template <typename T> struct FLam24 {
    const T *Ux, *Uy, *Uz, *Wx, *Wy, *Wz, *sx, *sy, *sz;
    __device__ void operator()(int64_t i, double *acc) const {
        T vx = Ux[i] - Wx[i], vy = Uy[i] - Wy[i], vz = Uz[i] - Wz[i];
        acc[0] += (double)vx * vx + (double)vy * vy + (double)vz * vz;
        acc[1] += (double)vx * sx[i] + (double)vy * sy[i] + (double)vz * sz[i];
    }
};

template <typename T> struct FLam35 {
    const T *Au, *b, *delta;
    __device__ void operator()(int64_t i, double *acc) const {
        T r = Au[i] - b[i];
        acc[0] += (double)r * r;
        acc[1] += (double)delta[i] * r;
    }
};

template <typename T> struct FShrink {
    const T *Ux, *Uy, *Uz, *sx, *sy, *sz;
    T beta;
    int iso;
    T *Wx, *Wy, *Wz;
    __device__ void operator()(int64_t i, double *acc) const {
        T ib = (T)1 / beta;
        T ux = Ux[i] - sx[i] / beta, uy = Uy[i] - sy[i] / beta, uz = Uz[i] - sz[i] / beta;
        if (!iso) {
            T tx = fabs(ux) - ib, ty = fabs(uy) - ib, tz = fabs(uz) - ib;
            tx = tx >= 0 ? tx : (T)0; ty = ty >= 0 ? ty : (T)0; tz = tz >= 0 ? tz : (T)0;
            Wx[i] = ux >= 0 ? tx : -tx;
            Wy[i] = uy >= 0 ? ty : -ty;
            Wz[i] = uz >= 0 ? tz : -tz;
            acc[0] += (double)tx + (double)ty + (double)tz;
        } else {
            T nrm = (T)sqrt((double)ux * ux + (double)uy * uy + (double)uz * uz);
            T sh = nrm - ib;
            if (sh > 0) {
                T f = sh / nrm;
                Wx[i] = ux * f; Wy[i] = uy * f; Wz[i] = uz * f;
                acc[0] += (double)sh;
            } else {
                Wx[i] = 0; Wy[i] = 0; Wz[i] = 0;
            }
        }
    }
};

template <typename T> struct FMlpSigma {
    const T *Ux, *Uy, *Uz, *Wx, *Wy, *Wz;
    T nb;
    T *sx, *sy, *sz;
    __device__ void operator()(int64_t i, double *acc) const {
        T vx = Ux[i] - Wx[i], vy = Uy[i] - Wy[i], vz = Uz[i] - Wz[i];
        T a = nb * vx + sx[i], b = nb * vy + sy[i], c = nb * vz + sz[i];
        sx[i] = a; sy[i] = b; sz[i] = c;
        acc[0] += (double)a * vx + (double)b * vy + (double)c * vz;
    }
};

template <typename T> struct FMlpDelta {
    const T *Au, *b;
    T nm;
    T *delta;
    __device__ void operator()(int64_t i, double *acc) const {
        T aub = Au[i] - b[i];
        T d = nm * aub + delta[i];
        delta[i] = d;
        acc[0] += (double)d * aub;
    }
};

template <typename T> struct FDiffNorm {
    const T *a, *b;
    __device__ void operator()(int64_t i, double *acc) const {
        T t = a[i] - b[i];
        acc[0] += (double)t * t;
        acc[1] += (double)a[i] * a[i];
    }
};

// Position of voxel i and its neighbours on the periodic grid; I: 32 bits
// where the volume allows (two 64-bit divisions a voxel would outweigh the
// memory traffic).
template <typename I> struct Grid3 {
    I p, q, r, pq;
    struct At {
        I i, y, x, z;
    };
    __device__ __forceinline__ At at(int64_t k) const {
        const I i = (I)k, c = i / p;
        return At{i, i - c * p, c % q, c / q};
    }
    __device__ __forceinline__ I up_y(const At &a) const { return a.y < p - 1 ? a.i + 1 : a.i - a.y; }
    __device__ __forceinline__ I up_x(const At &a) const { return a.x < q - 1 ? a.i + p : a.i - a.x * p; }
    __device__ __forceinline__ I up_z(const At &a) const { return a.z < r - 1 ? a.i + pq : a.i - a.z * pq; }
    __device__ __forceinline__ I dn_y(const At &a) const { return a.y == 0 ? a.i + (p - 1) : a.i - 1; }
    __device__ __forceinline__ I dn_x(const At &a) const { return a.x == 0 ? a.i + (q - 1) * p : a.i - p; }
    __device__ __forceinline__ I dn_z(const At &a) const { return a.z == 0 ? a.i + (r - 1) * pq : a.i - pq; }
};

// D^T (DU - W) at a voxel; v: DU - W there
template <typename T, typename I>
__device__ __forceinline__ T dt_of(const Grid3<I> &G, const typename Grid3<I>::At &a,
                                   const T *Ux, const T *Uy, const T *Uz, const T *Wx, const T *Wy,
                                   const T *Wz, T vx, T vy, T vz) {
    const I jy = G.dn_y(a), jx = G.dn_x(a), jz = G.dn_z(a);
    const T yp = Uy[jy] - Wy[jy], xp = Ux[jx] - Wx[jx], zp = Uz[jz] - Wz[jz];
    return yp - vy + xp - vx + zp - vz;
}

// the four sums of the exact step length: |D d|^2 per component, |d|^2
template <typename T, typename I> struct FStep {
    Grid3<I> G;
    const T *d;
    __device__ void operator()(int64_t k, double *acc) const {
        const auto a = G.at(k);
        const T t = d[a.i];
        const T dy = d[G.up_y(a)] - t, dx = d[G.up_x(a)] - t, dz = d[G.up_z(a)] - t;
        acc[0] += (double)dx * (double)dx;
        acc[1] += (double)dy * (double)dy;
        acc[2] += (double)dz * (double)dz;
        acc[3] += (double)t * (double)t;
    }
};

// after the products: lam2, lam4, g2 = D^T (DU - W), g = (A^T Au) - Atb
template <typename T, typename I> struct FGradient {
    Grid3<I> G;
    const T *Ux, *Uy, *Uz, *Wx, *Wy, *Wz, *sx, *sy, *sz, *Atb;
    T *g2, *g;     // g NULL: the A^T product was skipped
    __device__ void operator()(int64_t k, double *acc) const {
        const auto a = G.at(k);
        const I i = a.i;
        const T vx = Ux[i] - Wx[i], vy = Uy[i] - Wy[i], vz = Uz[i] - Wz[i];
        acc[0] += (double)vx * vx + (double)vy * vy + (double)vz * vz;
        acc[1] += (double)vx * sx[i] + (double)vy * sy[i] + (double)vz * sz[i];
        g2[i] = dt_of<T, I>(G, a, Ux, Uy, Uz, Wx, Wy, Wz, vx, vy, vz);
        if (g) g[i] = (T)-1 * Atb[i] + g[i];
    }
};

// the end of an iteration, W new: lam2, lam4, g2, the direction d, and the
// sums the next step length and the stopping test take: |d|^2, |U - Up|^2,
// |Up|^2, <U - Up, change of the gradient>
template <typename T, typename I> struct FUpdate {
    Grid3<I> G;
    const T *Ux, *Uy, *Uz, *Wx, *Wy, *Wz, *sx, *sy, *sz, *g, *gp, *g2p, *dts, *U, *Up;
    T mdb;
    T *g2, *d;
    __device__ void operator()(int64_t k, double *acc) const {
        const auto a = G.at(k);
        const I i = a.i;
        const T vx = Ux[i] - Wx[i], vy = Uy[i] - Wy[i], vz = Uz[i] - Wz[i];
        acc[0] += (double)vx * vx + (double)vy * vy + (double)vz * vz;
        acc[1] += (double)vx * sx[i] + (double)vy * sy[i] + (double)vz * sz[i];
        const T h = dt_of<T, I>(G, a, Ux, Uy, Uz, Wx, Wy, Wz, vx, vy, vz);
        g2[i] = h;
        const T gi = g[i], v = mdb * gi + h, di = v + dts[i];
        d[i] = di;
        acc[2] += (double)di * (double)di;
        const T up = Up[i], u = (T)-1 * up + U[i];
        const T dg = gi - gp[i], dg2 = h - g2p[i];
        acc[3] += (double)u * u;
        acc[4] += (double)up * (double)up;
        acc[5] += (double)u * (double)(dg2 + mdb * dg);
    }
};

// Block partials of K sums over n items by workgroup b of nb, a workgroup's K
// values side by side.
template <int K, typename F>
__device__ __forceinline__ void reduce_items(int64_t n, const F &f, int b, int nb,
                                             double *partials) {
    __shared__ double sh[K][4];
    double acc[K];
#pragma unroll
    for (int k = 0; k < K; ++k) acc[k] = 0.0;
    for (int64_t i = (int64_t)b * 256 + threadIdx.x; i < n; i += (int64_t)nb * 256) f(i, acc);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const double v = wave_sum(acc[k]);
        if (lane == 0) sh[k][wave] = v;
    }
    __syncthreads();
    if (threadIdx.x < K) {
        const double *w = sh[threadIdx.x];
        partials[(int64_t)b * K + threadIdx.x] = (w[0] + w[1]) + (w[2] + w[3]);
    }
}

template <int K, typename F>
__global__ __launch_bounds__(256) void k_reduce(int64_t n, F f, double *partials) {
    reduce_items<K>(n, f, blockIdx.x, gridDim.x, partials);
}

// Three reductions that do not depend on each other, one behind the other in
// the grid: a launch of its own for each costs 4 us of a 64^3 iteration's 70.
template <int K1, typename F1, int K2, typename F2, int K3, typename F3>
__global__ __launch_bounds__(256) void k_reduce3(int64_t n1, F1 f1, int nb1, int64_t n2, F2 f2,
                                                 int nb2, int64_t n3, F3 f3, int nb3,
                                                 double *partials) {
    const int b = blockIdx.x;
    if (b < nb1)
        reduce_items<K1>(n1, f1, b, nb1, partials);
    else if (b < nb1 + nb2)
        reduce_items<K2>(n2, f2, b - nb1, nb2, partials + (int64_t)K1 * nb1);
    else
        reduce_items<K3>(n3, f3, b - nb1 - nb2, nb3,
                         partials + (int64_t)K1 * nb1 + (int64_t)K2 * nb2);
}

// One workgroup a sum: adds its block partials in a fixed order and leaves
// the value in pinned host memory, then the ticket that says so.  (With the
// partials themselves in pinned memory the host read and added up to 9,700 of
// them an iteration while the device idled; see Sums.)
struct SumList {
    int first[kSumMax], stride[kSumMax], blocks[kSumMax];
};
__global__ __launch_bounds__(256) void k_sum_blocks(SumList L, const double *partials,
                                                    SumResult *out, uint64_t ticket) {
    __shared__ double sh[4];
    const int j = blockIdx.x, blocks = L.blocks[j], stride = L.stride[j];
    const double *p = partials + L.first[j];
    double v = 0.0;
    for (int b = threadIdx.x; b < blocks; b += 256) v += p[(int64_t)b * stride];
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        out[j].value = (sh[0] + sh[1]) + (sh[2] + sh[3]);
        __hip_atomic_store(&out[j].ticket, ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

static int sum_blocks(int64_t n) {
    return (int)std::min<int64_t>(std::max<int64_t>((n + 255) / 256, 1), kSumBlocks);
}

// room for the block partials of K more sums over n items
template <int K>
static double *place_sums(Sums &S, int64_t n) {
    tv3_ctx *ctx = S.ctx;
    if (!ctx->red_part.p) {
        ctx->red_part.alloc((size_t)kSumMax * kSumBlocks);
        ctx->red_host.alloc(kSumMax);
        for (int j = 0; j < kSumMax; ++j) ctx->red_host.p[j].ticket = 0;
    }
    TV3_REQUIRE(S.count + K <= kSumMax, TV3_E_INTERNAL, "too many sums at once");
    const int nb = sum_blocks(n);
    double *p = ctx->red_part.p + S.used;
    for (int k = 0; k < K; ++k) S.sum[S.count++] = {(int)S.used + k, K, nb};
    S.used += (size_t)K * nb;
    return p;
}

// queues the block partials of K sums over n items
template <int K, typename F>
static void queue_sums(Sums &S, int64_t n, const F &f) {
    double *p = place_sums<K>(S, n);
    hipLaunchKernelGGL((k_reduce<K, F>), dim3((unsigned)sum_blocks(n)), dim3(256), 0, S.s, n, f, p);
}

static inline void cpu_pause() {
#if defined(__x86_64__)
    __builtin_ia32_pause();
#endif
}

const double *Sums::fetch(bool drain) {
    SumList L{};
    for (int j = 0; j < count; ++j) {
        L.first[j] = sum[j].first;
        L.stride[j] = sum[j].stride;
        L.blocks[j] = sum[j].blocks;
    }
    const uint64_t ticket = ++ctx->red_ticket;
    SumResult *out = ctx->red_host.p;
    hipLaunchKernelGGL(k_sum_blocks, dim3((unsigned)count), dim3(256), 0, s, L, ctx->red_part.p, out,
                       ticket);
    TV3_HIP(hipGetLastError());
    auto landed = [&] {
        for (int j = 0; j < count; ++j)
            if (__atomic_load_n(&out[j].ticket, __ATOMIC_ACQUIRE) != ticket) return false;
        return true;
    };
    // a bounded watch of the tickets, then the stream's own wait (which also
    // reports a failed launch)
    bool there = false;
    if (!drain) {
        const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(2);
        while (!(there = landed()) && std::chrono::steady_clock::now() < until) cpu_pause();
    }
    if (!there) TV3_HIP(hipStreamSynchronize(s));
    for (int j = 0; j < count; ++j) value[j] = out[j].value;
    used = 0;
    count = 0;
    return value;
}

template <int K, typename F>
std::array<double, K> reduce_now(tv3_ctx *ctx, int64_t n, const F &f, hipStream_t s) {
    Sums S{ctx, s};
    queue_sums<K>(S, n, f);
    const double *v = S.fetch(/*drain=*/true);
    std::array<double, K> out{};
    for (int k = 0; k < K; ++k) out[k] = v[k];
    return out;
}

// a volume's grid with 32- or 64-bit indices
template <typename F>
static void with_grid(const int32_t d[3], F f) {
    const int64_t pq = (int64_t)d[0] * d[1];
    if (pq * d[2] < (int64_t(1) << 31))
        f(Grid3<int32_t>{d[0], d[1], d[2], (int32_t)pq});
    else
        f(Grid3<int64_t>{d[0], d[1], d[2], pq});
}

template <typename T, typename I>
__global__ __launch_bounds__(256) void k_descend(Grid3<I> G, int64_t n, T tau, int nonneg,
                                                 const T *__restrict__ U, const T *__restrict__ d,
                                                 T *__restrict__ V, T *__restrict__ Vx,
                                                 T *__restrict__ Vy, T *__restrict__ Vz) {
    const T a = -tau;
    auto moved = [&](I i) {
        const T v = a * d[i] + U[i];
        return nonneg && v < 0 ? (T)0 : v;
    };
    for (int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x; k < n; k += (int64_t)gridDim.x * 256) {
        const auto at = G.at(k);
        const T t = moved(at.i);
        V[at.i] = t;
        Vy[at.i] = moved(G.up_y(at)) - t;
        Vx[at.i] = moved(G.up_x(at)) - t;
        Vz[at.i] = moved(G.up_z(at)) - t;
    }
}

template <typename T>
void descend_step(const int32_t dims[3], double tau, bool nonneg, const T *U, const T *d, T *V,
                  T *Vx, T *Vy, T *Vz, hipStream_t s) {
    const int64_t n = (int64_t)dims[0] * dims[1] * dims[2];
    with_grid(dims, [&](auto G) {
        using I = decltype(G.p);
        hipLaunchKernelGGL((k_descend<T, I>), dim3(ew_blocks(n)), dim3(256), 0, s, G, n, (T)tau,
                           (int)nonneg, U, d, V, Vx, Vy, Vz);
    });
}

template <typename T>
void queue_step(Sums &S, const int32_t dims[3], const T *d) {
    with_grid(dims, [&](auto G) {
        using I = decltype(G.p);
        queue_sums<4>(S, (int64_t)dims[0] * dims[1] * dims[2], FStep<T, I>{G, d});
    });
}

template <typename T>
void queue_dot(Sums &S, int64_t n, const T *a, const T *b) {
    queue_sums<1>(S, n, FDot<T>{a, b});
}

template <typename T>
void queue_gradient(Sums &S, const PlainFields<T> &f, T *g, const T *Atb, int64_t m, const T *Au,
                    const T *b, const T *delta) {
    with_grid(f.dims, [&](auto G) {
        using I = decltype(G.p);
        queue_sums<2>(S, f.n, FGradient<T, I>{G, f.Ux, f.Uy, f.Uz, f.Wx, f.Wy, f.Wz, f.sx, f.sy,
                                              f.sz, Atb, f.g2, g});
    });
    queue_lam35<T>(S, m, Au, b, delta);
}

template <typename T>
void queue_trial(Sums &S, const PlainFields<T> &f, T *g, const T *Atb, int64_t m, const T *Au,
                 const T *b, const T *delta, const PlainFields<T> &next, int iso, double beta) {
    const FLam35<T> f2{Au, b, delta};
    const FShrink<T> f3{next.Ux, next.Uy, next.Uz, next.sx, next.sy, next.sz, (T)beta, iso,
                        next.Wx, next.Wy, next.Wz};
    with_grid(f.dims, [&](auto G) {
        using I = decltype(G.p);
        using F1 = FGradient<T, I>;
        const F1 f1{G, f.Ux, f.Uy, f.Uz, f.Wx, f.Wy, f.Wz, f.sx, f.sy, f.sz, Atb, f.g2, g};
        double *p = place_sums<2>(S, f.n);
        place_sums<2>(S, m);
        place_sums<1>(S, f.n);
        const int nb1 = sum_blocks(f.n), nb2 = sum_blocks(m);
        hipLaunchKernelGGL((k_reduce3<2, F1, 2, FLam35<T>, 1, FShrink<T>>),
                           dim3((unsigned)(2 * nb1 + nb2)), dim3(256), 0, S.s, f.n, f1, nb1, m, f2,
                           nb2, f.n, f3, nb1, p);
    });
}

template <typename T>
void queue_lam24(Sums &S, const PlainFields<T> &f) {
    queue_sums<2>(S, f.n, FLam24<T>{f.Ux, f.Uy, f.Uz, f.Wx, f.Wy, f.Wz, f.sx, f.sy, f.sz});
}

template <typename T>
void queue_lam35(Sums &S, int64_t m, const T *Au, const T *b, const T *delta) {
    queue_sums<2>(S, m, FLam35<T>{Au, b, delta});
}

template <typename T>
void queue_shrink(Sums &S, const PlainFields<T> &f, int iso, double beta) {
    queue_sums<1>(S, f.n, FShrink<T>{f.Ux, f.Uy, f.Uz, f.sx, f.sy, f.sz, (T)beta, iso, f.Wx, f.Wy,
                                     f.Wz});
}

template <typename T>
void queue_update(Sums &S, const PlainFields<T> &f, const T *g, const T *gp, const T *g2p,
                  const T *dts, const T *U, const T *Up, double mdb, T *d) {
    with_grid(f.dims, [&](auto G) {
        using I = decltype(G.p);
        queue_sums<6>(S, f.n, FUpdate<T, I>{G, f.Ux, f.Uy, f.Uz, f.Wx, f.Wy, f.Wz, f.sx, f.sy,
                                            f.sz, g, gp, g2p, dts, U, Up, (T)mdb, f.g2, d});
    });
}

template <typename T>
double shrink_host(tv3_ctx *ctx, int64_t n, int iso, const T *Ux, const T *Uy, const T *Uz,
                   const T *sx, const T *sy, const T *sz, double beta, T *Wx, T *Wy, T *Wz,
                   hipStream_t s) {
    return reduce_now<1>(ctx, n, FShrink<T>{Ux, Uy, Uz, sx, sy, sz, (T)beta, iso, Wx, Wy, Wz},
                         s)[0];
}
template <typename T>
double mlp_sigma(tv3_ctx *ctx, int64_t n, const T *Ux, const T *Uy, const T *Uz, const T *Wx,
                 const T *Wy, const T *Wz, double beta, T *sx, T *sy, T *sz, hipStream_t s) {
    return reduce_now<1>(ctx, n, FMlpSigma<T>{Ux, Uy, Uz, Wx, Wy, Wz, (T)(-beta), sx, sy, sz}, s)[0];
}
template <typename T>
double mlp_delta(tv3_ctx *ctx, int64_t m, const T *Au, const T *b, double mu, T *delta,
                 hipStream_t s) {
    return reduce_now<1>(ctx, m, FMlpDelta<T>{Au, b, (T)(-mu), delta}, s)[0];
}
template <typename T>
std::array<double, 2> diff_norm(tv3_ctx *ctx, int64_t n, const T *a, const T *b, hipStream_t s) {
    return reduce_now<2>(ctx, n, FDiffNorm<T>{a, b}, s);
}

#define TV3_INST(T)                                                                              \
    template void axpy3<T>(int64_t, T *, double, const T *, const T *, hipStream_t);            \
    template void grad<T>(int64_t, T *, double, const T *, const T *, const T *, hipStream_t);  \
    template void scale<T>(int64_t, T *, double, const T *, hipStream_t);                       \
    template void divide<T>(int64_t, T *, double, const T *, hipStream_t);                      \
    template void launch_D<T>(const int32_t *, const T *, T *, T *, T *, hipStream_t);          \
    template void launch_Dt<T>(const int32_t *, const T *, const T *, const T *, T *,           \
                               hipStream_t);                                                    \
    template double shrink_host<T>(tv3_ctx *, int64_t, int, const T *, const T *, const T *,    \
                                   const T *, const T *, const T *, double, T *, T *, T *,      \
                                   hipStream_t);                                                \
    template double mlp_sigma<T>(tv3_ctx *, int64_t, const T *, const T *, const T *,           \
                                 const T *, const T *, const T *, double, T *, T *, T *,        \
                                 hipStream_t);                                                  \
    template double mlp_delta<T>(tv3_ctx *, int64_t, const T *, const T *, double, T *,         \
                                 hipStream_t);                                                  \
    template std::array<double, 2> diff_norm<T>(tv3_ctx *, int64_t, const T *, const T *,       \
                                                hipStream_t);                                   \
    template void descend_step<T>(const int32_t *, double, bool, const T *, const T *, T *, T *, \
                                  T *, T *, hipStream_t);                                       \
    template void queue_step<T>(Sums &, const int32_t *, const T *);                            \
    template void queue_dot<T>(Sums &, int64_t, const T *, const T *);                          \
    template void queue_gradient<T>(Sums &, const PlainFields<T> &, T *, const T *, int64_t,    \
                                    const T *, const T *, const T *);                          \
    template void queue_trial<T>(Sums &, const PlainFields<T> &, T *, const T *, int64_t,       \
                                 const T *, const T *, const T *, const PlainFields<T> &, int,  \
                                 double);                                                       \
    template void queue_lam24<T>(Sums &, const PlainFields<T> &);                               \
    template void queue_lam35<T>(Sums &, int64_t, const T *, const T *, const T *);             \
    template void queue_shrink<T>(Sums &, const PlainFields<T> &, int, double);                 \
    template void queue_update<T>(Sums &, const PlainFields<T> &, const T *, const T *,         \
                                  const T *, const T *, const T *, const T *, double, T *);

TV3_INST(float)
TV3_INST(double)

}  // namespace tv3
