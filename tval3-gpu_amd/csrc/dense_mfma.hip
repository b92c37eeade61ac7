// dense_mfma.hip -- products of one dense BF16 matrix with up to 64
// right-hand sides on the matrix cores (v_mfma_f32_32x32x16_bf16).
//
// Y (R x G) = M (R x K) X (K x G), M BF16 in MFMA operand order (below),
// X FP32 column-major (right-hand side j at X + j ldx), Y FP32
// column-major (Y + j ldy), optionally minus a vector of the same layout.
// This is the dense operator's product (3d/mat_vec_mul_dense.h:25-73, gemv N
// and T) for several vectors at once: A x and A^T r each read a copy of A
// (M = A, M = A^T) built once on the device -- the dense counterpart of
// keeping a CSR and a CSC.
//
// Operand order: M is stored in blocks of 32 rows x 16 columns (1 KB), the
// blocks of a 32-row band consecutive along K; inside a block lane l's 8
// operands M[32 rb + l % 32][16 kb + 8 (l / 32) + e], e = 0..7, lie at
// (l * 8 + e).  One wavefront load of its A operands is then 1 KB of
// contiguous memory (eight whole cache lines) instead of 16 bytes from each
// of 32 rows K apart.
//
// Precision: A is BF16 by definition of the operator; each FP32 value of X
// is split into three BF16 terms, hi = bf16(x), mid = bf16(x - hi),
// lo = bf16(x - hi - mid), each multiplied into one FP32 accumulator (three
// MFMAs), so X enters with about 24 significant bits -- the products are as
// accurate as FP32 ones (two terms, 16 bits, leave a relative error near
// 2e-6 that TVAL3's step-size recursion amplifies).
//
// Work: a 512-thread workgroup owns 256 rows x 64 columns (wavefront w: rows
// 32w..32w+31, two 32 x 32 MFMA tiles) over one of S slices of K.  Per
// chunk of 64 K-values the workgroup converts X's 64 x 64 block to its three
// BF16 terms in LDS (read by all eight wavefronts); each lane loads its M operands
// (16 contiguous bytes of the operand-ordered copy) straight from memory,
// one chunk ahead.  The S partial tiles
// go to a row-major scratch; a second kernel sums them in a fixed order,
// subtracts, and writes Y column-major through an LDS transpose.
// Bound by reading M (and R x 64 partial sums per slice, written and read):
// 4096 x 16384, 64 columns, 132 -> 83 us for A X and A^T R together (M twice,
// 268 MB: 3.2 TB/s; the products alone 31-34 us each, 4.2 TB/s).  Converting X
// once per product into operand order (no conversion and one barrier here, a
// launch more) took 81 us, but 2-4 us more at 2048 x 8192 and below; M two
// chunks ahead at one workgroup a CU, workgroups of one XCD on the same slices
// of K: no change.
//
// MFMA operand layout (v_mfma_f32_32x32x16_bf16, checked on the device):
// lane l supplies A[l % 32][8 (l / 32) + e] and B[8 (l / 32) + e][l % 32],
// e = 0..7; accumulator r of lane l is D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32].
#include "tv3_internal.hpp"

namespace tv3 {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kRows = 256;   // rows per workgroup (8 wavefronts)
constexpr int kThreads = 512;
constexpr int kCols = 64;    // right-hand sides per launch
constexpr int kChunk = 64;   // K-values per LDS chunk
constexpr int kPadK = kChunk + 8;

__device__ __forceinline__ uint16_t bf16_rne(float x) {
    const uint32_t u = __float_as_uint(x);
    return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

__global__ __launch_bounds__(512, 4) void k_gemm_rhs(const uint16_t *__restrict__ M,
                                                  int64_t R, int64_t K, int each, int more,
                                                  const float *__restrict__ X, int64_t ldx,
                                                  int G, float *__restrict__ part,
                                                  const int32_t *gate) {
    if (gate && !*gate) return;
    __shared__ __attribute__((aligned(16))) uint16_t xh[kCols][kPadK];
    __shared__ __attribute__((aligned(16))) uint16_t xm[kCols][kPadK];
    __shared__ __attribute__((aligned(16))) uint16_t xl[kCols][kPadK];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t tiles = R / kRows;
    const int64_t tile = blockIdx.x % tiles;
    const int s = (int)(blockIdx.x / tiles);
    // slice s of K: `each` chunks, one more in the first `more` slices
    const int64_t nchunk = each + (s < more ? 1 : 0);
    const int64_t k_beg = ((int64_t)s * each + min(s, more)) * kChunk;
    // this wavefront's 32-row band of M in operand order, lane's 16 bytes
    const uint16_t *mrow = M + (tile * (kRows / 32) + wave) * (K / 16) * 512 + lane * 8;
    // X staging: thread t converts 8 values of column t / 8 (columns >= G
    // read column G - 1 and are zeroed: no branch around the loads)
    const int xc = t >> 3, xk = (t & 7) * 8;
    const float *xcol = X + (int64_t)(xc < G ? xc : G - 1) * ldx + xk;
    const float xon = xc < G ? 1.f : 0.f;
    f32x16 tot0 = {}, tot1 = {};
    // The next chunk's operands are requested while the current one is
    // multiplied: X's before the products, an operand of M as soon as its last
    // product is issued (into the same registers: two sets, and the totals,
    // would leave one workgroup a CU).
    auto load_a = [&](int64_t c, int st) {
        const int64_t kc = k_beg + min(c, nchunk - 1) * kChunk;   // clamped: in range
        return *reinterpret_cast<const bf16x8 *>(mrow + (kc / 16 + st) * 512);
    };
    float4 x0, x1;
    auto load_x = [&](int64_t c) {
        const float *p = xcol + k_beg + min(c, nchunk - 1) * kChunk;
        x0 = *reinterpret_cast<const float4 *>(p);
        x1 = *reinterpret_cast<const float4 *>(p + 4);
    };
    bf16x8 a[4];
    load_x(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int st = 0; st < 4; ++st) a[st] = load_a(0, st);
    for (int64_t c = 0; c < nchunk; ++c) {
        __syncthreads();   // the previous chunk's LDS operands have been read
        // the three BF16 terms of 8 values, packed two per word: 16-byte LDS stores
        {
            const float v[8] = {x0.x * xon, x0.y * xon, x0.z * xon, x0.w * xon,
                                x1.x * xon, x1.y * xon, x1.z * xon, x1.w * xon};
            uint32_t ph[4], pm[4], pl[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                ph[e] = pm[e] = pl[e] = 0;
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const float w = v[2 * e + u];
                    const uint32_t h = bf16_rne(w);
                    const float r1 = w - __uint_as_float(h << 16);
                    const uint32_t md = bf16_rne(r1);
                    const float r2 = r1 - __uint_as_float(md << 16);
                    ph[e] |= h << (16 * u);
                    pm[e] |= md << (16 * u);
                    pl[e] |= (uint32_t)bf16_rne(r2) << (16 * u);
                }
            }
            *reinterpret_cast<uint4 *>(&xh[xc][xk]) = make_uint4(ph[0], ph[1], ph[2], ph[3]);
            *reinterpret_cast<uint4 *>(&xm[xc][xk]) = make_uint4(pm[0], pm[1], pm[2], pm[3]);
            *reinterpret_cast<uint4 *>(&xl[xc][xk]) = make_uint4(pl[0], pl[1], pl[2], pl[3]);
        }
        __builtin_amdgcn_sched_barrier(0);
        load_x(c + 1);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        // a chunk's sums (64 products a term) start at zero and are added to
        // the totals: a chain as long as a whole slice of K loses bits
        f32x16 acc0 = {}, acc1 = {};
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            const int kk = 16 * st + 8 * (lane >> 5);
            const int c0 = lane & 31, c1 = 32 + (lane & 31);
            auto term = [&](const uint16_t (*xt)[kPadK]) {
                const bf16x8 b0 = *reinterpret_cast<const bf16x8 *>(&xt[c0][kk]);
                const bf16x8 b1 = *reinterpret_cast<const bf16x8 *>(&xt[c1][kk]);
                acc0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[st], b0, acc0, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[st], b1, acc1, 0, 0, 0);
            };
            term(xl);          // smallest terms first: the large ones are added last
            term(xm);
            term(xh);
            a[st] = load_a(c + 1, st);
        }
        tot0 += acc0;
        tot1 += acc1;
        // issue order: kAhead operand reads lead the matrix instructions, each
        // of which is followed by one more read; a step's load of M goes out
        // as soon as its operand is free.  Left alone the compiler reads an
        // operand, waits, multiplies, and sinks the loads to the loop's end.
        constexpr int kAhead = 4;
        __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);
#pragma unroll
        for (int k = 0; k < 24; ++k) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (k < 24 - kAhead) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            if (k % 6 == 5) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        }
    }
    // partial tile, row-major [s][row][64]
    float *out = part + ((int64_t)s * R + tile * kRows + wave * 32) * kCols;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int i = 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        out[(int64_t)i * kCols + (lane & 31)] = tot0[r];
        out[(int64_t)i * kCols + 32 + (lane & 31)] = tot1[r];
    }
}

// Y[j ldy + row] = sum_s part[s][row][j] (- sub[j ldy + row]), j < G: one
// workgroup per 8 rows, a thread sums every other partial of four columns of
// a row (fixed order), eight loads in flight; the halves meet in LDS, read
// back with rows consecutive.  (32 rows a workgroup and one chain of S loads
// a thread took 11 us at S = 16, and 25 us of a whole 35 us product at 1024 x
// 4096 and S = 64.)
__global__ __launch_bounds__(256) void k_gemm_reduce(const float *__restrict__ part, int64_t R,
                                                     int S, int G, float *__restrict__ Y,
                                                     int64_t ldy, const float *__restrict__ sub,
                                                     const int32_t *gate) {
    if (gate && !*gate) return;
    __shared__ float tile[2][8][kCols + 1];
    const int t = threadIdx.x;
    const int64_t r0 = (int64_t)blockIdx.x * 8;
    const int c = (t & 15) * 4, row = (t >> 4) & 7, half = t >> 7;
    const float *p = part + (r0 + row) * kCols + c;
    float4 v = make_float4(0, 0, 0, 0);
    auto add = [&v](const float4 &w) {
        v.x += w.x; v.y += w.y; v.z += w.z; v.w += w.w;
    };
    int s = half;
    for (; s + 14 < S; s += 16) {
        float4 w[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            w[i] = *reinterpret_cast<const float4 *>(p + (int64_t)(s + 2 * i) * R * kCols);
#pragma unroll
        for (int i = 0; i < 8; ++i) add(w[i]);
    }
    for (; s < S; s += 2) add(*reinterpret_cast<const float4 *>(p + (int64_t)s * R * kCols));
    float *o = &tile[half][row][c];
    o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
    __syncthreads();
    const int rr = t & 7;
#pragma unroll
    for (int cc = t >> 3; cc < kCols; cc += 32) {
        if (cc >= G) break;
        const int64_t q = (int64_t)cc * ldy + r0 + rr;
        const float w = tile[0][rr][cc] + tile[1][rr][cc];
        Y[q] = sub ? w - sub[q] : w;
    }
}

// Operand-ordered copy of M = A (trans = 0, R = m, K = n) or M = A^T
// (trans = 1, R = n, K = m) from a column-major m x n BF16 matrix A (leading
// dimension lda): thread (block, lane) writes lane's 8 operands of one
// 32 x 16 block (16 bytes)
__global__ __launch_bounds__(256) void k_operand_order_bf16(const uint16_t *__restrict__ A,
                                                            int64_t lda, int trans, int64_t R,
                                                            int64_t K, uint16_t *__restrict__ Mt) {
    const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t nkb = K / 16;
    if (g >= (R / 32) * nkb * 64) return;
    const int lane = (int)(g & 63);
    const int64_t blk = g >> 6, rb = blk / nkb, kb = blk % nkb;
    const int64_t row = 32 * rb + (lane & 31), col = 16 * kb + 8 * (lane >> 5);
    uint16_t v[8];
    if (trans) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = A[row * lda + col + e];   // column row of A
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = A[(col + e) * lda + row];
    }
    uint4 w;
    w.x = v[0] | ((uint32_t)v[1] << 16); w.y = v[2] | ((uint32_t)v[3] << 16);
    w.z = v[4] | ((uint32_t)v[5] << 16); w.w = v[6] | ((uint32_t)v[7] << 16);
    *reinterpret_cast<uint4 *>(Mt + g * 8) = w;
}

}  // namespace

int gemm_rhs_rows() { return kRows; }

bool gemm_rhs_shape_ok(int64_t R, int64_t K, int splits) {
    return R > 0 && K > 0 && R % kRows == 0 && splits > 0 && K % ((int64_t)splits * kChunk) == 0;
}

void gemm_rhs(const uint16_t *M, int64_t R, int64_t K, const float *X, int64_t ldx, int G,
              float *Y, int64_t ldy, const float *sub, int splits, float *part, hipStream_t s,
              const int32_t *gate) {
    TV3_REQUIRE(G > 0 && G <= kCols, TV3_E_ARG, "1 to 64 right-hand sides per product");
    TV3_REQUIRE(R > 0 && R % kRows == 0 && K % kChunk == 0 && splits > 0 && splits <= K / kChunk,
                TV3_E_SHAPE,
                "dense multi-RHS products need rows a multiple of 256 and K a multiple of 64, "
                "with at least 64 values for each split");
    TV3_REQUIRE(ldx % 4 == 0, TV3_E_SHAPE,
                "dense multi-RHS products need 16-byte aligned right-hand sides");
    const unsigned grid = (unsigned)((R / kRows) * splits);
    const int64_t chunks = K / kChunk;
    hipLaunchKernelGGL(k_gemm_rhs, dim3(grid), dim3(kThreads), 0, s, M, R, K, (int)(chunks / splits),
                       (int)(chunks % splits), X, ldx, G, part, gate);
    hipLaunchKernelGGL(k_gemm_reduce, dim3((unsigned)(R / 8)), dim3(256), 0, s, part, R, splits,
                       G, Y, ldy, sub, gate);
}

size_t gemm_rhs_scratch(int64_t R, int splits) { return (size_t)splits * R * kCols; }

void dense_operand_order(tv3_op *op, hipStream_t s) {
    if (op->dense_oN.p) return;
    TV3_REQUIRE(op->dtype == TV3_BF16, TV3_E_FORMAT,
                "dense multi-RHS products take BF16 matrices");
    TV3_REQUIRE(op->m % 32 == 0 && op->n % 32 == 0, TV3_E_SHAPE,
                "dense multi-RHS products need rows and columns multiples of 32");
    const size_t bytes = (size_t)op->m * op->n * 2;
    DevBuf<uint8_t> oN(bytes), oT(bytes);
    const int64_t threads = op->m * op->n / 8;
    const unsigned grid = (unsigned)((threads + 255) / 256);
    hipLaunchKernelGGL(k_operand_order_bf16, dim3(grid), dim3(256), 0, s,
                       (const uint16_t *)op->dense.p, op->lda, 0, op->m, op->n,
                       (uint16_t *)oN.p);
    hipLaunchKernelGGL(k_operand_order_bf16, dim3(grid), dim3(256), 0, s,
                       (const uint16_t *)op->dense.p, op->lda, 1, op->n, op->m,
                       (uint16_t *)oT.p);
    TV3_HIP(hipGetLastError());
    TV3_HIP(hipStreamSynchronize(s));    // the next product may run on another stream
    op->dense_oN = std::move(oN);
    op->dense_oT = std::move(oT);
}

}  // namespace tv3
