// spmv.hip -- CSR products y = A x and y = A^T x (via the CSC, stored as the
// CSR of A^T) for gfx950, plus the device scan and the stable transpose.
//
// Semantics follow the single-GPU sparse operator of the reference
// (3d/mat_vec_mul_sparse.h:1703-1780: csrmv with alpha = 1, beta = 0 on the
// CSR for N and on the CSC arrays for T); the kernels are new.
//
// Kernel shape: a group of L lanes (L a power of two, 2..64) owns one row.
// Lanes stride over the row's entries, so one group reads L consecutive
// (col, val) pairs per step and a 64-wide wavefront reads 64/L rows' worth of
// consecutive memory: the col/val streams are fully coalesced whatever L is.
// x is gathered (it stays in L2 / MALL); the group sum is a butterfly over L
// lanes.  L is chosen from the mean row length or by the autotuner.  That
// form serves FP64 vectors on matrices with long rows and what set_lanes or
// the autotuner picks; a new operator's products run over row blocks.
#include <algorithm>

#include "spmv_stream.hpp"

namespace tv3 {

template <typename V> __device__ __forceinline__ float ldw(const V *p, int64_t k);
template <> __device__ __forceinline__ float ldw<float>(const float *p, int64_t k) { return p[k]; }
template <> __device__ __forceinline__ float ldw<__half>(const __half *p, int64_t k) {
    return __half2float(p[k]);
}
template <> __device__ __forceinline__ float ldw<__hip_bfloat16>(const __hip_bfloat16 *p, int64_t k) {
    return __bfloat162float(p[k]);
}
__device__ __forceinline__ double ldw64(const double *p, int64_t k) { return p[k]; }
__device__ __forceinline__ double ldw64(const float *p, int64_t k) { return (double)p[k]; }

// Acc = float: FP32 accumulation (the fast path).  Acc = double: each row
// sum is formed in FP64 and rounded once, which restates the oracle's
// rounding (used by the reference-shaped solver).
template <int L, typename V, typename Acc>
__global__ __launch_bounds__(256) void k_csr_f32(int64_t rows, const int32_t *__restrict__ ptr,
                                                 const int32_t *__restrict__ ind,
                                                 const V *__restrict__ val,
                                                 const float *__restrict__ x,
                                                 float *__restrict__ y) {
    const int64_t bid = xcd_remap(blockIdx.x, gridDim.x);
    const int64_t row = (bid * 256 + threadIdx.x) / L;
    const int lane = threadIdx.x & (L - 1);
    if (row >= rows) return;          // whole groups leave together (L divides 256)
    const int beg = ptr[row], end = ptr[row + 1];
    Acc s = 0;
    int k = beg + lane;
    // two independent chains keep two gathers in flight per lane
    Acc s2 = 0;
    for (; k + L < end; k += 2 * L) {
        const int c0 = ind[k], c1 = ind[k + L];
        const Acc w0 = (Acc)ldw<V>(val, k), w1 = (Acc)ldw<V>(val, k + L);
        s = fma(w0, (Acc)x[c0], s);
        s2 = fma(w1, (Acc)x[c1], s2);
    }
    if (k < end) s = fma((Acc)ldw<V>(val, k), (Acc)x[ind[k]], s);
    s = lane_sum<L>(s + s2);
    if (lane == 0) y[row] = (float)s;
}

template <int L, typename V>
__global__ __launch_bounds__(256) void k_csr_f64(int64_t rows, const int32_t *__restrict__ ptr,
                                                 const int32_t *__restrict__ ind,
                                                 const V *__restrict__ val,
                                                 const double *__restrict__ x,
                                                 double *__restrict__ y) {
    const int64_t row = ((int64_t)blockIdx.x * 256 + threadIdx.x) / L;
    const int lane = threadIdx.x & (L - 1);
    if (row >= rows) return;
    const int beg = ptr[row], end = ptr[row + 1];
    double s = 0.0;
    for (int k = beg + lane; k < end; k += L) s = fma(ldw64(val, k), x[ind[k]], s);
    s = lane_sum<L>(s);
    if (lane == 0) y[row] = s;
}

int default_lanes(int64_t rows, int64_t nnz) {
    double avg = rows > 0 ? (double)nnz / (double)rows : 0.0;
    int L = 2;
    while (L < 64 && L < avg / 2.0) L <<= 1;
    return L;
}

template <typename V, typename Acc>
static void launch_f32(const SparseRows &S, const float *x, float *y, hipStream_t s, int L) {
    const V *val = reinterpret_cast<const V *>(S.val.p);
    const int64_t threads = S.rows * L;
    const unsigned blocks = (unsigned)((threads + 255) / 256);
    if (blocks == 0) return;
#define TV3_CASE(LL)                                                                      \
    case LL:                                                                              \
        hipLaunchKernelGGL((k_csr_f32<LL, V, Acc>), dim3(blocks), dim3(256), 0, s, S.rows,\
                           S.ptr.p, S.ind.p, val, x, y);                                  \
        break;
    switch (L) {
        TV3_CASE(2) TV3_CASE(4) TV3_CASE(8) TV3_CASE(16) TV3_CASE(32) TV3_CASE(64)
    default: throw tv3_error(TV3_E_ARG, "lanes per row must be a power of two in [2, 64]");
    }
#undef TV3_CASE
    TV3_HIP(hipGetLastError());
}

template <typename V>
static void launch_f64(const SparseRows &S, const double *x, double *y, hipStream_t s, int L) {
    const V *val = reinterpret_cast<const V *>(S.val.p);
    const int64_t threads = S.rows * L;
    const unsigned blocks = (unsigned)((threads + 255) / 256);
    if (blocks == 0) return;
#define TV3_CASE(LL)                                                                      \
    case LL:                                                                              \
        hipLaunchKernelGGL((k_csr_f64<LL, V>), dim3(blocks), dim3(256), 0, s, S.rows,     \
                           S.ptr.p, S.ind.p, val, x, y);                                  \
        break;
    switch (L) {
        TV3_CASE(2) TV3_CASE(4) TV3_CASE(8) TV3_CASE(16) TV3_CASE(32) TV3_CASE(64)
    default: throw tv3_error(TV3_E_ARG, "lanes per row must be a power of two in [2, 64]");
    }
#undef TV3_CASE
    TV3_HIP(hipGetLastError());
}

// Wavefront blocks: at most kWave rows and kWaveBlk entries, or one longer row.
constexpr int kWave = 64, kWaveBlk = 256;
static bool wave_blocks(const SparseRows &S) { return S.blk_nnz == kWaveBlk; }

// The sum of w x over a row's entries of one lane, products unrounded.  A
// chain's first product is rounded, so the up to four entries of a lane of 64
// (rows of 65 to 256 entries) make one chain; with fewer lanes two shorter
// chains err less.  RMS error against k_csr_f64's order, 2 to 256 entries a
// row, random weights and values: 0.91 to 1.01 (with rounded products 1.00 to
// 1.11).
template <int NB>
__device__ __forceinline__ double row_fma(const double2 *wx, int a, int e, int lane, int L) {
    double s0 = 0, s1 = 0;
    for (int k = a + lane; k < e; k += 4 * L) {
        double2 v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = wx[min(k + i * L, NB - 1)];
        const bool in1 = k + L < e, in2 = k + 2 * L < e, in3 = k + 3 * L < e;
        s0 = fma(v[0].x, v[0].y, s0);
        if (L == kWave) {
            s0 = in1 ? fma(v[1].x, v[1].y, s0) : s0;
            s0 = in2 ? fma(v[2].x, v[2].y, s0) : s0;
            s0 = in3 ? fma(v[3].x, v[3].y, s0) : s0;
        } else {
            s1 = in1 ? fma(v[1].x, v[1].y, s1) : s1;
            s0 = in2 ? fma(v[2].x, v[2].y, s0) : s0;
            s1 = in3 ? fma(v[3].x, v[3].y, s1) : s1;
        }
    }
    return s0 + s1;
}

// Row blocks for one wavefront each: the block's (col, val) pairs are read
// with unit stride, its products go to the wavefront's part of LDS, and
// 1 << lg lanes sum each row.  Nothing waits for another wavefront, so the
// phases of neighbouring blocks overlap; eight times smaller blocks than
// k_csr_stream's also fill the chip more evenly when few are left.  A longer
// row (a voxel next to a transducer) is summed lane by lane, J gathers in
// flight.
//
// Bound by the line fills of the gathers (L2 -> L1, 128 B each: 23.5M for
// either product at 128^3, 28 TB/s in A^T) and, where x outgrows an L2 slice,
// by its misses (A: 4.3M, 22 TB/s of fills; A^T 1.9M).  us, against 2048-entry
// blocks of a 256-thread workgroup: 64^3 voxels x 65,536 rays FP32 weights
// A^T 27.0 -> 18.0, A 17.2 -> 17.0; 128^3 x 262,144 FP16 A^T 130 -> 107,
// A 149 -> 148, FP64 A^T 298 -> 187, A 300 -> 260 (k_csr_f64); A in natural
// block order (order_blocks).
//
// Acc = double also serves FP32 vectors whose row sums are rounded once: their
// products fit 53 bits.  An FP64 vector's do not, so LDS then holds weights and
// gathered values, and the row sums are fused multiply-adds.
template <typename V, typename X, typename Acc>
__global__ __launch_bounds__(256) void k_csr_wave(const BlkDesc *__restrict__ desc,
                                                  const int32_t *__restrict__ ptr,
                                                  const int32_t *__restrict__ ind,
                                                  const V *__restrict__ val,
                                                  const X *__restrict__ x, X *__restrict__ y,
                                                  int nblk) {
    constexpr int J = kWaveBlk / kWave;
    constexpr bool kUnrounded = std::is_same_v<X, double>;
    using Term = std::conditional_t<kUnrounded, double2, Acc>;
    __shared__ Term terms[256 / kWave][kWaveBlk];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int b = xcd_remap(blockIdx.x, gridDim.x) * (256 / kWave) + wave;
    if (b >= nblk) return;
    Term *term = terms[wave];
    const int t = threadIdx.x & (kWave - 1);
    const BlkDesc d = desc[b];
    const int L = 1 << d.lg, rr = t >> d.lg, lane = t & (L - 1);
    const bool has = rr < d.nr;
    const int row = d.r0 + (has ? rr : d.nr - 1);
    const int end = d.p0 + d.len;
    const int a = ptr[row], e = ptr[row + 1];
    V w[J];
    // J entries of this lane from entry k0 on, clamped to the block's last.
    // Loads return in order, so with the weights requested first a gather
    // starts when its entry's streams are in; earlier gathers crowd out the
    // streams of other wavefronts.  A and A^T in turn, the matrices from HBM,
    // 128^3, us (columns first -> weights first): FP16 310 -> 277, FP32 301 ->
    // 296.
    Acc p[J];
    auto entries = [&](int k0) {
#pragma unroll
        for (int j = 0; j < J; ++j) w[j] = val[min(k0 + j * kWave + t, end - 1)];
        __builtin_amdgcn_sched_barrier(0);
        int c[J];
#pragma unroll
        for (int j = 0; j < J; ++j) c[j] = ind[min(k0 + j * kWave + t, end - 1)];
#pragma unroll
        for (int j = 0; j < J; ++j) p[j] = (Acc)x[c[j]];
    };
    if (d.len > 0) entries(d.p0);
    auto weight = [](V v) {
        if constexpr (std::is_same_v<V, double>) return v;
        else return (Acc)to_f32(v);
    };
    Acc s = 0;
    if (d.len <= kWaveBlk) {
        if (d.len > 0) {
#pragma unroll
            for (int j = 0; j < J; ++j) {
                if constexpr (kUnrounded) term[j * kWave + t] = make_double2(weight(w[j]), p[j]);
                else term[j * kWave + t] = weight(w[j]) * p[j];
            }
        }
        // the wavefront's own LDS operations complete in order
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if constexpr (kUnrounded) {
            if (has) s = row_fma<kWaveBlk>(term, a - d.p0, e - d.p0, lane, L);
        } else {
            if (has) s = row_sum<kWaveBlk>(term, a - d.p0, e - d.p0, lane, L);
        }
    } else {
        for (int k0 = d.p0;;) {
#pragma unroll
            for (int j = 0; j < J; ++j)
                if (k0 + j * kWave + t < end) s = fma(weight(w[j]), p[j], s);
            k0 += kWaveBlk;
            if (k0 >= end) break;
            entries(k0);
        }
    }
    s = lane_sum(s, L);
    if (has && lane == 0) y[row] = (X)s;
}

template <typename V, typename X, typename Acc>
static void launch_wave(const SparseRows &S, const X *x, X *y, hipStream_t s) {
    if (S.nblk == 0) return;
    hipLaunchKernelGGL((k_csr_wave<V, X, Acc>), dim3((unsigned)((S.nblk + 3) / 4)), dim3(256), 0, s,
                       S.desc.p, S.ptr.p, S.ind.p, reinterpret_cast<const V *>(S.val.p), x, y,
                       (int)S.nblk);
    TV3_HIP(hipGetLastError());
}

static std::vector<int32_t> row_pointers(tv3_ctx *ctx, const SparseRows &S) {
    std::vector<int32_t> ptr(S.rows + 1);
    TV3_HIP(hipMemcpyAsync(ptr.data(), S.ptr.p, sizeof(int32_t) * (S.rows + 1),
                           hipMemcpyDeviceToHost, ctx->stream));
    TV3_HIP(hipStreamSynchronize(ctx->stream));
    return ptr;
}

static std::vector<BlkDesc> row_blocks(tv3_ctx *ctx, SparseRows &S, int blk_nnz,
                                       const std::vector<int32_t> &ptr,
                                       const std::vector<int64_t> *starts) {
    const int threads = blk_nnz == kWaveBlk ? kWave : 256;
    std::vector<int32_t> blk;
    blk.reserve(S.nnz / (blk_nnz / 2) + S.rows / threads + 2);
    int64_t start = 0;
    size_t si = 0;   // next forced block start
    blk.push_back(0);
    for (int64_t r = 0; r < S.rows; ++r) {
        while (starts && si < starts->size() && (*starts)[si] < r) ++si;
        const bool forced = starts && si < starts->size() && (*starts)[si] == r;
        // close the current block before row r if adding it would overflow
        if (r > start &&
            (forced || (int64_t)ptr[r + 1] - ptr[start] > blk_nnz || r - start >= threads)) {
            blk.push_back((int32_t)r);
            start = r;
        }
    }
    blk.push_back((int32_t)S.rows);
    S.nblk = (int64_t)blk.size() - 1;
    std::vector<BlkDesc> d = make_blk_desc(blk, ptr.data(), nullptr, threads);
    S.desc.alloc(d.size());
    TV3_HIP(hipMemcpyAsync(S.desc.p, d.data(), sizeof(BlkDesc) * d.size(), hipMemcpyHostToDevice,
                           ctx->stream));
    TV3_HIP(hipStreamSynchronize(ctx->stream));
    S.blk_nnz = blk_nnz;
    return d;
}

void build_row_blocks(tv3_ctx *ctx, SparseRows &S, int blk_nnz,
                      const std::vector<int64_t> *starts) {
    row_blocks(ctx, S, blk_nnz, row_pointers(ctx, S), starts);
}

// Where a block's first row runs: the sixteenths of the columns that its ends
// lie in, and its middle entry's 4096th (20 bits).
constexpr int kKeyBits = 20, kMiddleBits = 12;
__global__ __launch_bounds__(256) void k_block_keys(int64_t nblk, int64_t cols,
                                                    const BlkDesc *__restrict__ desc,
                                                    const int32_t *__restrict__ ptr,
                                                    const int32_t *__restrict__ ind,
                                                    uint32_t *__restrict__ key) {
    const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (b >= nblk) return;
    const int r = desc[b].r0, p0 = ptr[r], p1 = ptr[r + 1];
    uint32_t v = 0;
    if (p0 < p1) {
        const int64_t i = ind[p0], j = ind[p1 - 1], k = ind[p0 + (p1 - p0) / 2];
        const uint32_t lo = (uint32_t)(16 * min(i, j) / cols), hi = (uint32_t)(16 * max(i, j) / cols);
        v = lo << 16 | hi << kMiddleBits | (uint32_t)((k << kMiddleBits) / cols);
    }
    key[b] = v;
}

// Blocks in the order of their keys (stable): the blocks that an XCD runs one
// after the other then gather from the same parts of x, whatever order the
// rays come in; the matrix and y stay as they are.  Worth it where x (FP32) is
// larger than an XCD's L2: A x, us, natural order -> this, 128^3 voxels x
// 262,144 rays FP16 148 -> 135, FP64 260 -> 220, 112^3 x 262,144 FP16 118 ->
// 112, 128^3 x 65,536 FP16 40.5 -> 38; below it the scattered streams cost
// more than the gathers gain (96^3 x 147,456 FP32 54 -> 56).
//
// And only where more than half of the blocks have their ends in other
// sixteenths than the block before: rows that are local already, and rows
// whose ends say nothing, pay for the scattered streams and gain nothing.
// 128^3 columns, FP16 / FP64 vectors with FP32 weights, changes, us natural ->
// ordered: shuffled rays 99 % 194 -> 139 / 323 -> 194; by emitter 94 % 148 ->
// 134 / 236 -> 185; by receiver 52 % 128 -> 123 / 182 -> 171; in bundles of
// 4 x 4 neighbours 34 % 122 -> 122 / 166 -> 170, of 8 x 8 28 % 115 -> 121 /
// 160 -> 169; 100 random columns a row 0.6 % 253 -> 262 / 361 -> 368.
constexpr int64_t kOrderedCols = (int64_t(4) << 20) / sizeof(float);
static void order_blocks(tv3_ctx *ctx, SparseRows &S, const std::vector<BlkDesc> &d) {
    const int64_t nb = S.nblk;
    if (nb < 2) return;
    hipStream_t s = ctx->stream;
    DevBuf<uint32_t> key(nb);
    hipLaunchKernelGGL(k_block_keys, dim3((unsigned)((nb + 255) / 256)), dim3(256), 0, s, nb, S.cols,
                       S.desc.p, S.ptr.p, S.ind.p, key.p);
    TV3_HIP(hipGetLastError());
    std::vector<uint32_t> k(nb);
    TV3_HIP(hipMemcpyAsync(k.data(), key.p, sizeof(uint32_t) * nb, hipMemcpyDeviceToHost, s));
    TV3_HIP(hipStreamSynchronize(s));
    int64_t changes = 0;
    for (int64_t b = 1; b < nb; ++b) changes += k[b] >> kMiddleBits != k[b - 1] >> kMiddleBits;
    if (2 * changes <= nb) return;
    std::vector<int32_t> from(nb), to(nb);
    for (int64_t b = 0; b < nb; ++b) from[b] = (int32_t)b;
    constexpr int kDigit = kKeyBits / 2, kBins = 1 << kDigit;
    for (int shift = 0; shift < kKeyBits; shift += kDigit) {
        std::vector<int32_t> at(kBins + 1, 0);
        for (int64_t b = 0; b < nb; ++b) ++at[(k[b] >> shift & (kBins - 1)) + 1];
        for (int i = 0; i < kBins; ++i) at[i + 1] += at[i];
        for (int64_t b = 0; b < nb; ++b) to[at[k[from[b]] >> shift & (kBins - 1)]++] = from[b];
        from.swap(to);
    }
    std::vector<BlkDesc> o(d);
    for (int64_t b = 0; b < nb; ++b) o[b] = d[from[b]];
    TV3_HIP(hipMemcpyAsync(S.desc.p, o.data(), sizeof(BlkDesc) * o.size(), hipMemcpyHostToDevice, s));
    TV3_HIP(hipStreamSynchronize(s));
}

// Wavefront blocks, unless a row is so long that one wavefront would still
// sum it when the others are done (16 rounds of gathers): then 2048-entry
// workgroup blocks.  Voxels next to a transducer are crossed by about 1,000
// rays of 262,144.  A^T, us, 256 / 512 entries a wavefront: 64^3 voxels
// 18.0 / 20.7, 96^3 49 / 49, 128^3 107 / 112.
void build_default_blocks(tv3_ctx *ctx, SparseRows &S, bool measurements) {
    const std::vector<int32_t> ptr = row_pointers(ctx, S);
    int32_t longest = 0;
    for (int64_t r = 0; r < S.rows; ++r) longest = std::max(longest, ptr[r + 1] - ptr[r]);
    const std::vector<BlkDesc> d =
        row_blocks(ctx, S, longest <= 16 * kWaveBlk ? kWaveBlk : 2048, ptr, nullptr);
    if (measurements && wave_blocks(S) && S.cols > kOrderedCols) order_blocks(ctx, S, d);
}

std::vector<BlkDesc> make_blk_desc(const std::vector<int32_t> &blk, const int32_t *ptr,
                                   const std::vector<int32_t> *pad_start, int threads) {
    const size_t nb = blk.empty() ? 0 : blk.size() - 1;
    std::vector<BlkDesc> d(nb + 1);
    for (size_t b = 0; b < nb; ++b) {
        BlkDesc &e = d[b];
        e.r0 = blk[b];
        e.nr = blk[b + 1] - blk[b];
        // kernels serve row r0 + min(lane group, nr - 1): a block needs a row
        TV3_REQUIRE(e.nr > 0, TV3_E_FORMAT, "row block without rows");
        e.p0 = ptr[blk[b]];
        e.len = ptr[blk[b + 1]] - e.p0;
        e.q0 = pad_start ? (*pad_start)[b] : e.p0;
        int lg = 6;
        while (lg > 0 && (1 << lg) * e.nr > threads) --lg;
        e.lg = lg;
        e.pad0 = e.pad1 = 0;
    }
    BlkDesc &z = d[nb];
    z.r0 = nb ? blk[nb] : 0;
    z.nr = z.len = z.lg = z.pad0 = z.pad1 = 0;
    z.p0 = z.q0 = nb ? ptr[blk[nb]] : 0;
    if (pad_start && nb) z.q0 = (*pad_start)[nb];
    return d;
}

void spmv_csr(const SparseRows &S, const float *x, float *y, hipStream_t s, int lanes,
              bool acc64) {
    if (!lanes && wave_blocks(S)) {
        switch (S.vtype) {
        case TV3_F32:
            acc64 ? launch_wave<float, float, double>(S, x, y, s)
                  : launch_wave<float, float, float>(S, x, y, s);
            return;
        case TV3_F16:
            acc64 ? launch_wave<__half, float, double>(S, x, y, s)
                  : launch_wave<__half, float, float>(S, x, y, s);
            return;
        case TV3_BF16:
            acc64 ? launch_wave<__hip_bfloat16, float, double>(S, x, y, s)
                  : launch_wave<__hip_bfloat16, float, float>(S, x, y, s);
            return;
        default: throw tv3_error(TV3_E_FORMAT, "FP32 products need F32, F16 or BF16 values");
        }
    }
    if (!lanes && S.blk_nnz) {
        if (acc64) launch_stream_any<double>(S, x, EpiStore<double>{y}, s);
        else launch_stream_any<float>(S, x, EpiStore<float>{y}, s);
        TV3_HIP(hipGetLastError());
        return;
    }
    int L = lanes ? lanes : (S.lanes ? S.lanes : default_lanes(S.rows, S.nnz));
    switch (S.vtype) {
    case TV3_F32:
        acc64 ? launch_f32<float, double>(S, x, y, s, L) : launch_f32<float, float>(S, x, y, s, L);
        break;
    case TV3_F16:
        acc64 ? launch_f32<__half, double>(S, x, y, s, L) : launch_f32<__half, float>(S, x, y, s, L);
        break;
    case TV3_BF16:
        acc64 ? launch_f32<__hip_bfloat16, double>(S, x, y, s, L)
              : launch_f32<__hip_bfloat16, float>(S, x, y, s, L);
        break;
    default: throw tv3_error(TV3_E_FORMAT, "FP32 products need F32, F16 or BF16 values");
    }
}

void spmv_csr(const SparseRows &S, const double *x, double *y, hipStream_t s, int lanes,
              bool) {
    if (!lanes && wave_blocks(S)) {
        switch (S.vtype) {
        case TV3_F64: launch_wave<double, double, double>(S, x, y, s); return;
        case TV3_F32: launch_wave<float, double, double>(S, x, y, s); return;
        default: throw tv3_error(TV3_E_FORMAT, "FP64 products need F64 or F32 values");
        }
    }
    int L = lanes ? lanes : (S.lanes ? S.lanes : default_lanes(S.rows, S.nnz));
    switch (S.vtype) {
    case TV3_F64: launch_f64<double>(S, x, y, s, L); break;
    case TV3_F32: launch_f64<float>(S, x, y, s, L); break;
    default: throw tv3_error(TV3_E_FORMAT, "FP64 products need F64 or F32 values");
    }
}

// ------------------------------------------------- several right-hand sides
// Xt[i][j] = X[i + j ldx] for j < G, 0 for G <= j < KT: one gather then brings
// an entry's values for all columns.
template <int KT>
__global__ __launch_bounds__(256) void k_columns_to_rows(int64_t n, int G,
                                                         const float *__restrict__ X, int64_t ldx,
                                                         float *__restrict__ Xt) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float v[KT];
#pragma unroll
    for (int j = 0; j < KT; ++j) v[j] = j < G ? X[i + j * ldx] : 0.f;
#pragma unroll
    for (int j = 0; j < KT; j += 4)
        *reinterpret_cast<float4 *>(Xt + i * KT + j) = make_float4(v[j], v[j + 1], v[j + 2], v[j + 3]);
}

__device__ __forceinline__ float4 operator*(float a, const float4 &b) {
    return make_float4(a * b.x, a * b.y, a * b.z, a * b.w);
}

// row_sum of four columns at once: each column's additions in row_sum's order
template <int NB>
__device__ __forceinline__ float4 row_sum4(const float4 *prod, int a, int e, int lane, int L) {
    float4 s0 = make_float4(0, 0, 0, 0), s1 = s0;
    for (int k = a + lane; k < e; k += 4 * L) {
        float4 v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = prod[min(k + i * L, NB - 1)];
            if (i > 0 && k + i * L >= e) v[i] = make_float4(0, 0, 0, 0);
        }
        s0.x += v[0].x + v[2].x; s0.y += v[0].y + v[2].y;
        s0.z += v[0].z + v[2].z; s0.w += v[0].w + v[2].w;
        s1.x += v[1].x + v[3].x; s1.y += v[1].y + v[3].y;
        s1.z += v[1].z + v[3].z; s1.w += v[1].w + v[3].w;
    }
    return make_float4(s0.x + s1.x, s0.y + s1.y, s0.z + s1.z, s0.w + s1.w);
}

// k_csr_stream (W = 256) or k_csr_wave (W = 64) for KT columns: a row block's
// entries are read once, KT / 4 neighbouring lanes gather one entry's KT
// values (one line look-up serves them), the products go to LDS, and W
// threads per four columns sum the rows.  Every column is summed as the
// kernel for one vector sums it (same bits).  Bound
// by the gathers of Xt: at 64^3 voxels and 65,536 rays, 8 columns, FP32
// weights, Xt included, A 41 us and A^T 39 us (2048-entry blocks 43 and 68),
// against eight launches of 17 and 18 us.
template <int NB, int KT, int W, typename V>
__global__ __launch_bounds__(W * KT / 4) void k_csr_multi(const BlkDesc *__restrict__ desc,
                                                       const int32_t *__restrict__ ptr,
                                                       const int32_t *__restrict__ ind,
                                                       const V *__restrict__ val,
                                                       const float *__restrict__ Xt,
                                                       float *__restrict__ Y, int64_t ldy, int G) {
    constexpr int Q = KT / 4;                // quads of columns
    __shared__ float4 prod[Q][NB];
    const BlkDesc d = desc[xcd_remap(blockIdx.x, gridDim.x)];
    const int t = threadIdx.x % W, q2 = threadIdx.x / W;         // phase 2: thread, quad
    const int L = 1 << d.lg, rr = t >> d.lg, lane = t & (L - 1);
    const bool has = rr < d.nr;
    const int row = d.r0 + (has ? rr : d.nr - 1);
    if (d.len <= NB) {
        constexpr int J = NB / W;
        const int a = ptr[row] - d.p0, e = ptr[row + 1] - d.p0;
        if (d.len > 0) {
            const int q = threadIdx.x % Q, slot = threadIdx.x / Q, last = d.p0 + d.len - 1;
            int c[J];
            V w[J];                          // weights first: see k_csr_wave
#pragma unroll
            for (int j = 0; j < J; ++j) w[j] = val[min(d.p0 + j * W + slot, last)];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < J; ++j) c[j] = ind[min(d.p0 + j * W + slot, last)];
#pragma unroll
            for (int j = 0; j < J; ++j)
                prod[q][j * W + slot] =
                    to_f32(w[j]) * *reinterpret_cast<const float4 *>(Xt + (int64_t)c[j] * KT + 4 * q);
        }
        __syncthreads();
        float4 s = make_float4(0, 0, 0, 0);
        if (has) s = row_sum4<NB>(prod[q2], a, e, lane, L);
        const float o[4] = {lane_sum(s.x, L), lane_sum(s.y, L), lane_sum(s.z, L), lane_sum(s.w, L)};
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (has && lane == 0 && 4 * q2 + j < G) Y[row + (4 * q2 + j) * ldy] = o[j];
    } else if constexpr (W == kWave) {
        // one row longer than NB, summed as k_csr_wave does
        float s[4] = {};
        for (int k = d.p0 + t; k < d.p0 + d.len; k += kWave) {
            const float w = ld_weight<V>(val, k);
            const float *x = Xt + (int64_t)ind[k] * KT + 4 * q2;
#pragma unroll
            for (int j = 0; j < 4; ++j) s[j] = fma(w, x[j], s[j]);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            s[j] = lane_sum<kWave>(s[j]);
            if (t == 0 && 4 * q2 + j < G) Y[row + (4 * q2 + j) * ldy] = s[j];
        }
    } else {
        // one row longer than NB
        float s[4] = {};
        for (int k = d.p0 + t; k < d.p0 + d.len; k += 256) {
            const float w = ld_weight<V>(val, k);
            const float *x = Xt + (int64_t)ind[k] * KT + 4 * q2;
#pragma unroll
            for (int j = 0; j < 4; ++j) s[j] += w * x[j];
        }
        float *sh = reinterpret_cast<float *>(prod);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            s[j] = lane_sum<64>(s[j]);
            if ((t & 63) == 0) sh[4 * (4 * q2 + j) + (t >> 6)] = s[j];
        }
        __syncthreads();
        const int g = threadIdx.x;
        if (g < G) Y[d.r0 + g * ldy] = (sh[4 * g] + sh[4 * g + 1]) + (sh[4 * g + 2] + sh[4 * g + 3]);
    }
}

bool spmv_multi_ok(const SparseRows &S) {
    return S.blk_nnz != 0 && (S.vtype == TV3_F32 || S.vtype == TV3_F16 || S.vtype == TV3_BF16);
}

size_t spmv_multi_scratch(const SparseRows &S) { return (size_t)S.cols * 8; }

template <int NB, int KT, int W, typename V>
static void launch_blocks(const SparseRows &S, int G, const float *xt, float *Y, int64_t ldy,
                          hipStream_t s) {
    hipLaunchKernelGGL((k_csr_multi<NB, KT, W, V>), dim3((unsigned)S.nblk), dim3(W * KT / 4), 0, s,
                       S.desc.p, S.ptr.p, S.ind.p, reinterpret_cast<const V *>(S.val.p), xt, Y, ldy,
                       G);
}

template <int KT, typename V>
static void launch_multi(const SparseRows &S, int G, const float *xt, float *Y, int64_t ldy,
                         hipStream_t s) {
    switch (S.blk_nnz) {
    case kWaveBlk: launch_blocks<kWaveBlk, KT, kWave, V>(S, G, xt, Y, ldy, s); return;
    case 1024: launch_blocks<1024, KT, 256, V>(S, G, xt, Y, ldy, s); return;
    case 2048: launch_blocks<2048, KT, 256, V>(S, G, xt, Y, ldy, s); return;
    case 4096:           // 64 KB of products for four columns
        if constexpr (KT == 4) {
            launch_blocks<4096, KT, 256, V>(S, G, xt, Y, ldy, s);
            return;
        }
    default: throw tv3_error(TV3_E_ARG, "stream block size must be 1024, 2048 or 4096");
    }
}

template <int KT>
static void multi(const SparseRows &S, int G, const float *X, int64_t ldx, float *Y, int64_t ldy,
                  float *xt, hipStream_t s) {
    hipLaunchKernelGGL(k_columns_to_rows<KT>, dim3((unsigned)((S.cols + 255) / 256)), dim3(256), 0,
                       s, S.cols, G, X, ldx, xt);
    if (S.nblk == 0) return;
    switch (S.vtype) {
    case TV3_F32: launch_multi<KT, float>(S, G, xt, Y, ldy, s); break;
    case TV3_F16: launch_multi<KT, __half>(S, G, xt, Y, ldy, s); break;
    default: launch_multi<KT, __hip_bfloat16>(S, G, xt, Y, ldy, s); break;
    }
}

void spmv_multi(const SparseRows &S, int nrhs, const float *X, int64_t ldx, float *Y, int64_t ldy,
                float *xt, hipStream_t s) {
    if (nrhs > 4 && S.blk_nnz <= 2048) {
        multi<8>(S, nrhs, X, ldx, Y, ldy, xt, s);
    } else {
        multi<4>(S, std::min(nrhs, 4), X, ldx, Y, ldy, xt, s);
        if (nrhs > 4) multi<4>(S, nrhs - 4, X + 4 * ldx, ldx, Y + 4 * ldy, ldy, xt, s);
    }
    TV3_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ scan
// Three passes: per-block sums of 1024 elements, a single-block carried scan
// of the block sums, then the per-block exclusive scan with its offset.
__global__ __launch_bounds__(256) void k_block_sums(const int32_t *cnt, int64_t n,
                                                    int64_t *bsum) {
    __shared__ int64_t sh[256];
    int64_t base = (int64_t)blockIdx.x * 1024;
    int64_t v = 0;
    for (int j = 0; j < 4; ++j) {
        int64_t i = base + threadIdx.x * 4 + j;
        if (i < n) v += cnt[i];
    }
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if (threadIdx.x < off) sh[threadIdx.x] += sh[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) bsum[blockIdx.x] = sh[0];
}

__global__ __launch_bounds__(256) void k_scan_sums(int64_t *bsum, int64_t nb, int64_t *total) {
    // exclusive scan of nb values, 256 at a time with a running carry
    __shared__ int64_t sh[256];
    int64_t carry = 0;
    for (int64_t base = 0; base < nb; base += 256) {
        int64_t i = base + threadIdx.x;
        int64_t v = i < nb ? bsum[i] : 0;
        sh[threadIdx.x] = v;
        __syncthreads();
        for (int off = 1; off < 256; off <<= 1) {
            int64_t t = threadIdx.x >= off ? sh[threadIdx.x - off] : 0;
            __syncthreads();
            sh[threadIdx.x] += t;
            __syncthreads();
        }
        if (i < nb) bsum[i] = carry + sh[threadIdx.x] - v;
        int64_t blocktot = sh[255];
        __syncthreads();
        carry += blocktot;
    }
    if (threadIdx.x == 0) *total = carry;
}

__global__ __launch_bounds__(256) void k_block_scan(const int32_t *cnt, int64_t n,
                                                    const int64_t *boff, int32_t *out) {
    __shared__ int64_t sh[256];
    int64_t base = (int64_t)blockIdx.x * 1024 + threadIdx.x * 4;
    int64_t v[4], tsum = 0;
    for (int j = 0; j < 4; ++j) {
        v[j] = (base + j < n) ? cnt[base + j] : 0;
        tsum += v[j];
    }
    sh[threadIdx.x] = tsum;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        int64_t t = threadIdx.x >= off ? sh[threadIdx.x - off] : 0;
        __syncthreads();
        sh[threadIdx.x] += t;
        __syncthreads();
    }
    int64_t run = boff[blockIdx.x] + sh[threadIdx.x] - tsum;
    for (int j = 0; j < 4; ++j) {
        if (base + j < n) out[base + j] = (int32_t)run;
        run += v[j];
    }
}

__global__ void k_set_last(int32_t *out, int64_t n, const int64_t *total) {
    out[n] = (int32_t)*total;
}

int64_t exclusive_scan_i32(tv3_ctx *ctx, const int32_t *cnt, int32_t *out, int64_t n) {
    hipStream_t s = ctx->stream;
    int64_t nb = (n + 1023) / 1024;
    DevBuf<int64_t> bsum(nb + 1);
    int64_t *total = bsum.p + nb;
    if (nb > 0) {
        hipLaunchKernelGGL(k_block_sums, dim3((unsigned)nb), dim3(256), 0, s, cnt, n, bsum.p);
        hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(256), 0, s, bsum.p, nb, total);
        hipLaunchKernelGGL(k_block_scan, dim3((unsigned)nb), dim3(256), 0, s, cnt, n, bsum.p,
                           out);
    } else {
        TV3_HIP(hipMemsetAsync(total, 0, sizeof(int64_t), s));
    }
    hipLaunchKernelGGL(k_set_last, dim3(1), dim3(1), 0, s, out, n, total);
    TV3_HIP(hipGetLastError());
    int64_t h = 0;
    TV3_HIP(hipMemcpyAsync(&h, total, sizeof(int64_t), hipMemcpyDeviceToHost, s));
    TV3_HIP(hipStreamSynchronize(s));
    TV3_REQUIRE(h <= INT32_MAX, TV3_E_SHAPE, "more than 2^31-1 entries: int32 indices overflow");
    return h;
}

// ------------------------------------------------------------------ transpose
__global__ void k_col_count(const int32_t *ind, int64_t nnz, int32_t *cnt) {
    int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < nnz) atomicAdd(&cnt[ind[k]], 1);
}

template <int VB>
__global__ void k_scatter(int64_t rows, const int32_t *ptr, const int32_t *ind,
                          const uint8_t *val, int32_t *cursor, int32_t *orow, uint8_t *oval) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= rows) return;
    for (int k = ptr[i]; k < ptr[i + 1]; ++k) {
        int pos = atomicAdd(&cursor[ind[k]], 1);
        orow[pos] = (int32_t)i;
#pragma unroll
        for (int b = 0; b < VB; ++b) oval[(int64_t)pos * VB + b] = val[(int64_t)k * VB + b];
    }
}

// Sort each column's entries by row: makes the transpose independent of the
// atomic arrival order.  Entries are packed as (row << 32 | value bits)
// keys.  Columns of up to 64 entries: one thread, insertion sort in private
// memory; longer columns (rays start inside the volume, so a transducer's
// voxel can hold thousands of entries): one workgroup each, bitonic sort in
// LDS.
template <int VB>
__device__ __forceinline__ uint64_t pack_key(const int32_t *row, const uint8_t *val, int64_t k) {
    uint32_t v = 0;
#pragma unroll
    for (int t = 0; t < VB; ++t) v |= (uint32_t)val[k * VB + t] << (8 * t);
    return ((uint64_t)(uint32_t)row[k] << 32) | v;
}
template <int VB>
__device__ __forceinline__ void unpack_key(uint64_t key, int32_t *row, uint8_t *val, int64_t k) {
    row[k] = (int32_t)(key >> 32);
    const uint32_t v = (uint32_t)key;
#pragma unroll
    for (int t = 0; t < VB; ++t) val[k * VB + t] = (uint8_t)(v >> (8 * t));
}

template <int VB>
__global__ void k_sort_cols(int64_t cols, const int32_t *cptr, int32_t *row, uint8_t *val,
                            int32_t *long_list, int32_t *long_count) {
    int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= cols) return;
    const int b = cptr[j], e = cptr[j + 1], len = e - b;
    if (len < 2) return;
    if (len > 64) {
        long_list[atomicAdd(long_count, 1)] = (int32_t)j;
        return;
    }
    uint64_t key[64];
    for (int a = 0; a < len; ++a) key[a] = pack_key<VB>(row, val, b + a);
    for (int a = 1; a < len; ++a) {
        const uint64_t k = key[a];
        int c = a - 1;
        while (c >= 0 && key[c] > k) { key[c + 1] = key[c]; --c; }
        key[c + 1] = k;
    }
    for (int a = 0; a < len; ++a) unpack_key<VB>(key[a], row, val, b + a);
}

// 8-byte values (FP64 operators): in-place insertion sort by row.
__global__ void k_sort_cols_f64(int64_t cols, const int32_t *cptr, int32_t *row, double *val) {
    int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= cols) return;
    const int b = cptr[j], e = cptr[j + 1];
    for (int a = b + 1; a < e; ++a) {
        const int32_t r = row[a];
        const double v = val[a];
        int c = a - 1;
        while (c >= b && row[c] > r) { row[c + 1] = row[c]; val[c + 1] = val[c]; --c; }
        row[c + 1] = r;
        val[c + 1] = v;
    }
}

constexpr int kLongSortCap = 8192;   // LDS keys per workgroup (64 KiB)

template <int VB>
__global__ __launch_bounds__(256) void k_sort_long(const int32_t *list, const int32_t *cptr,
                                                   int32_t *row, uint8_t *val) {
    __shared__ uint64_t key[kLongSortCap];
    const int j = list[blockIdx.x];
    const int b = cptr[j], len = cptr[j + 1] - b;
    int P = 1;
    while (P < len) P <<= 1;
    for (int a = threadIdx.x; a < P; a += 256)
        key[a] = a < len ? pack_key<VB>(row, val, b + a) : ~0ull;
    __syncthreads();
    for (int k = 2; k <= P; k <<= 1) {
        for (int jj = k >> 1; jj > 0; jj >>= 1) {
            for (int i = threadIdx.x; i < P; i += 256) {
                const int l = i ^ jj;
                if (l > i) {
                    const uint64_t x = key[i], y = key[l];
                    const bool up = (i & k) == 0;
                    if ((x > y) == up) { key[i] = y; key[l] = x; }
                }
            }
            __syncthreads();
        }
    }
    for (int a = threadIdx.x; a < len; a += 256) unpack_key<VB>(key[a], row, val, b + a);
}

void build_transpose(tv3_ctx *ctx, const SparseRows &A, SparseRows &AT) {
    hipStream_t s = ctx->stream;
    AT.rows = A.cols;
    AT.cols = A.rows;
    AT.nnz = A.nnz;
    AT.vtype = A.vtype;
    AT.ptr.alloc(AT.rows + 1);
    AT.ind.alloc(A.nnz > 0 ? A.nnz : 1);
    const size_t vb = dtype_size(A.vtype);
    AT.val.alloc((A.nnz > 0 ? A.nnz : 1) * vb);
    DevBuf<int32_t> cnt(AT.rows + 1);
    TV3_HIP(hipMemsetAsync(cnt.p, 0, cnt.bytes(), s));
    if (A.nnz > 0)
        hipLaunchKernelGGL(k_col_count, dim3((unsigned)((A.nnz + 255) / 256)), dim3(256), 0, s,
                           A.ind.p, A.nnz, cnt.p);
    exclusive_scan_i32(ctx, cnt.p, AT.ptr.p, AT.rows);
    TV3_HIP(hipMemcpyAsync(cnt.p, AT.ptr.p, sizeof(int32_t) * AT.rows, hipMemcpyDeviceToDevice, s));
    unsigned gb = (unsigned)((A.rows + 255) / 256), gc = (unsigned)((AT.rows + 255) / 256);
    if (A.nnz > 0 && vb == 8) {
        hipLaunchKernelGGL(k_scatter<8>, dim3(gb), dim3(256), 0, s, A.rows, A.ptr.p, A.ind.p,
                           A.val.p, cnt.p, AT.ind.p, AT.val.p);
        hipLaunchKernelGGL(k_sort_cols_f64, dim3(gc), dim3(256), 0, s, AT.rows, AT.ptr.p, AT.ind.p,
                           reinterpret_cast<double *>(AT.val.p));
    } else if (A.nnz > 0) {
        DevBuf<int32_t> list(AT.rows > 0 ? AT.rows : 1), lcount(1);
        TV3_HIP(hipMemsetAsync(lcount.p, 0, sizeof(int32_t), s));
        if (vb == 2) {
            hipLaunchKernelGGL(k_scatter<2>, dim3(gb), dim3(256), 0, s, A.rows, A.ptr.p, A.ind.p,
                               A.val.p, cnt.p, AT.ind.p, AT.val.p);
            hipLaunchKernelGGL(k_sort_cols<2>, dim3(gc), dim3(256), 0, s, AT.rows, AT.ptr.p,
                               AT.ind.p, AT.val.p, list.p, lcount.p);
        } else {
            hipLaunchKernelGGL(k_scatter<4>, dim3(gb), dim3(256), 0, s, A.rows, A.ptr.p, A.ind.p,
                               A.val.p, cnt.p, AT.ind.p, AT.val.p);
            hipLaunchKernelGGL(k_sort_cols<4>, dim3(gc), dim3(256), 0, s, AT.rows, AT.ptr.p,
                               AT.ind.p, AT.val.p, list.p, lcount.p);
        }
        int32_t nlong = 0;
        TV3_HIP(hipMemcpyAsync(&nlong, lcount.p, sizeof(int32_t), hipMemcpyDeviceToHost, s));
        TV3_HIP(hipStreamSynchronize(s));
        if (nlong > 0) {
            // every long column must fit the LDS sort
            std::vector<int32_t> lst(nlong), cp(AT.rows + 1);
            TV3_HIP(hipMemcpy(lst.data(), list.p, sizeof(int32_t) * nlong, hipMemcpyDeviceToHost));
            TV3_HIP(hipMemcpy(cp.data(), AT.ptr.p, sizeof(int32_t) * (AT.rows + 1),
                              hipMemcpyDeviceToHost));
            for (int32_t j : lst)
                TV3_REQUIRE(cp[j + 1] - cp[j] <= kLongSortCap, TV3_E_SHAPE,
                            "a column holds more than 8192 entries (device transpose limit)");
            if (vb == 2)
                hipLaunchKernelGGL(k_sort_long<2>, dim3(nlong), dim3(256), 0, s, list.p, AT.ptr.p,
                                   AT.ind.p, AT.val.p);
            else
                hipLaunchKernelGGL(k_sort_long<4>, dim3(nlong), dim3(256), 0, s, list.p, AT.ptr.p,
                                   AT.ind.p, AT.val.p);
        }
    }
    TV3_HIP(hipGetLastError());
    TV3_HIP(hipStreamSynchronize(s));
    AT.lanes = default_lanes(AT.rows, AT.nnz);
}

}  // namespace tv3
