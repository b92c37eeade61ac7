// solver_plain.hip -- the reference-shaped TVAL3 loop on the device, with
// host-side scalars, in the order of
// 3d/tval3_gpu_3d.cpp:1088-1345 (get_g :366-572, get_tau :577-666, descend
// :671-701, update_g :706-818, min_u :823-891, get_gradient :896-919,
// shrinkage :924-960, update_W :965-1029, update_mlp :1034-1083).
//
// Differences from the reference, all deliberate:
//  * one stream, so no cross-stream races (the reference's get_g/update_g/
//    update_W read V on a stream that did not wait for its producer);
//  * lam2/lam4 use all three components with sigma in X,Y,Z order;
//  * inner products accumulate in FP64 (block partials summed in a fixed
//    order), scalars are FP64, and every entry of a product
//    A x is summed in FP64 and rounded once, so the FP32 iterates restate
//    the oracle's rounding instead of the accumulation order of a library;
//  * vector kernels are compiled without FP contraction (a*x+y rounds
//    twice, as written);
//  * vector operations between two host decisions share kernels (descend + D;
//    the gradient parts with lam2, lam4; shrinkage; the update of W's
//    consequences with every sum the next decision needs), each element
//    computed and rounded as by one kernel per operation; an iteration
//    without backtracking waits for the device once, and the previous iterate
//    is kept by exchanging buffers (64^3 voxels, 65,536 rays: 70 us an
//    iteration against 270 us with one kernel per operation and a wait per
//    inner product);
//  * the work vectors stay with the context (the reference allocates and
//    frees 3 n-vectors inside get_g/update_g/update_W/update_mlp);
//  * the A^T-skip heuristic (:398-468) leaves a skipped g as A^T(last Au)
//    - Atb; the reference subtracts Atb a second time from the stale g
//    (:463-467 then :565-567).
// This path is the parity anchor and the baseline the fused path is
// measured against.
#include <cmath>
#include <cstring>
#include <limits>
#include <utility>

#include "vec.hpp"

namespace tv3 {

namespace {

template <typename T>
struct PlainState {
    tv3_ctx *ctx;
    tv3_op *op;
    const tv3_opts *o;
    hipStream_t s;
    int32_t dims[3];
    int64_t n, m;
    double mu, beta, muDbeta, f, lam1, lam2, lam3, lam4, lam5;
    T *delta, *sx, *sy, *sz, *dU, *dUx, *dUy, *dUz, *Atb, *dAu, *dg, *dg2, *Ad, *DtsAtd, *rcdU,
        *bs, *lastAu, *dlast;
    // the iterate and what follows from it (0), and the previous one's (1)
    T *U[2], *Ux[2], *Uy[2], *Uz[2], *g[2], *g2[2], *Au[2];
    // W, D^T (DU - W) for it and the direction: in use (0; g2[0]) and next
    T *Wx[2], *Wy[2], *Wz[2], *d[2], *g2_next;
    double dd = 0, uu = 0, upup = 0, ug = 0;   // |d|^2, |U - Up|^2, |Up|^2, <U - Up, dgrad>
    int64_t nN = 0, nT = 0;
    int cur_init = 0;        // A^T-skip state (:155-157)
    double cur_skip = 0.0;
    bool last_mul = true;    // the last get_g multiplied by A^T

    void alloc() {
        // DtsAtd, sigma and delta start at zero (:1128-1139)
        T **nv[] = {&DtsAtd, &sx, &sy, &sz, &dU, &dUx, &dUy, &dUz, &Wx[0], &Wx[1], &Wy[0],
                    &Wy[1], &Wz[0], &Wz[1], &Atb, &d[0], &d[1], &dg, &dg2, &g2_next, &rcdU, &U[0], &U[1], &Ux[0], &Ux[1], &Uy[0], &Uy[1], &Uz[0], &Uz[1],
                    &g[0], &g[1], &g2[0], &g2[1]};
        T **mv[] = {&delta, &dAu, &Ad, &bs, &lastAu, &dlast, &Au[0], &Au[1]};
        const size_t cn = sizeof(nv) / sizeof(nv[0]), cm = sizeof(mv) / sizeof(mv[0]);
        // pad each vector to 256 bytes
        auto pad = [](int64_t k) { return (k + 63) / 64 * 64; };
        const size_t need = sizeof(T) * (cn * pad(n) + cm * pad(m));
        if (ctx->plain_ws.bytes() < need) ctx->plain_ws.alloc(need);
        T *p = reinterpret_cast<T *>(ctx->plain_ws.p);
        for (size_t k = 0; k < cn; ++k) { *nv[k] = p; p += pad(n); }
        for (size_t k = 0; k < cm; ++k) { *mv[k] = p; p += pad(m); }
        TV3_HIP(hipMemsetAsync(DtsAtd, 0, sizeof(T) * 4 * pad(n), s));
        TV3_HIP(hipMemsetAsync(delta, 0, sizeof(T) * m, s));
        // the skip rule compares with lastAu before the first product fills it
        TV3_HIP(hipMemsetAsync(lastAu, 0, sizeof(T) * m, s));
    }
    PlainFields<T> fields() {
        return {dims, n, Ux[0], Uy[0], Uz[0], Wx[0], Wy[0], Wz[0], sx, sy, sz, g2[0]};
    }
    // the iterate becomes the previous one
    void turn() {
        for (auto *v : {U, Ux, Uy, Uz, g, g2, Au}) std::swap(v[0], v[1]);
    }
    void copy(T *dst, const T *src, int64_t k) {
        TV3_HIP(hipMemcpyAsync(dst, src, sizeof(T) * k, hipMemcpyDeviceToDevice, s));
    }
    void A(bool trans, const T *x, T *y) {
        op_apply(op, trans, x, y, s, /*acc64=*/true);
        (trans ? nT : nN)++;
    }
    double fval() const { return lam1 + beta / 2 * lam2 + mu / 2 * lam3 - lam4 - lam5; }

    void set_f(const double *v) {      // lam2, lam4, lam3, lam5
        lam2 = v[0]; lam4 = v[1]; lam3 = v[2]; lam5 = v[3];
        f = fval();
    }
    // :366-572; force: the initial and the fallback call (:1148, :880).  With
    // ahead the sums of update_W are queued behind and returned too.
    const double *get_g(Sums &S, bool force, bool ahead) {
        A(false, U[0], Au[0]);
        bool mul = true;
        if (o->skipMulRatio != 0.0) {
            // relative change of Au since the last A^T product (:398-412)
            axpy3<T>(m, dlast, -1.0, lastAu, Au[0], s);
            Sums R{ctx, s};
            queue_dot<T>(R, m, dlast, dlast);
            queue_dot<T>(R, m, Au[0], Au[0]);
            const double *v = R.fetch();
            const double rel = std::sqrt(v[0]) / std::sqrt(v[1]);
            if (force) {
                cur_skip = 0.0;
            } else if ((uint32_t)cur_init < o->numInitIterations) {
                ++cur_init;
                cur_skip = 0.0;
            } else if (cur_skip < 1.0) {
                cur_skip += o->skipMulRatio;
            } else if (rel > o->maxRelativeChange) {
                // Au moved too far: multiply
            } else {
                cur_skip -= 1.0;
                mul = false;
            }
            if (mul) copy(lastAu, Au[0], m);
        }
        if (mul) A(true, Au[0], g[0]);
        else copy(g[0], g[1], n);          // g stays as it was
        T *gm = mul ? g[0] : nullptr;
        if (ahead) {
            queue_trial<T>(S, fields(), gm, Atb, m, Au[0], bs, delta, next_fields(), iso(), beta);
            queue_next(S);
        } else {
            queue_gradient<T>(S, fields(), gm, Atb, m, Au[0], bs, delta);
        }
        last_mul = mul;
        const double *v = S.fetch();
        set_f(v);
        return v + 4;
    }
    // exact step length along d (:577-640); leaves |d|^2
    double first_tau() {
        A(false, d[0], Ad);
        Sums S{ctx, s};
        queue_step<T>(S, dims, d[0]);
        queue_dot<T>(S, m, Ad, Ad);
        const double *v = S.fetch();
        const double dDd = v[0] + v[1] + v[2];
        dd = v[3];
        return std::fabs(dd / (dDd + muDbeta * v[4]));
    }
    const double *descend(Sums &S, double tau, bool force, bool ahead) {
        descend_step<T>(dims, tau, o->nonneg != 0, U[1], d[0], U[0], Ux[0], Uy[0], Uz[0], s);
        return get_g(S, force, ahead);
    }
    void update_g(double alpha) {
        axpy3<T>(n, g[0], alpha, dg, g[1], s);
        axpy3<T>(n, g2[0], alpha, dg2, g2[1], s);
        axpy3<T>(n, U[0], alpha, dU, U[1], s);
        axpy3<T>(m, Au[0], alpha, dAu, Au[1], s);
        axpy3<T>(n, Ux[0], alpha, dUx, Ux[1], s);
        axpy3<T>(n, Uy[0], alpha, dUy, Uy[1], s);
        axpy3<T>(n, Uz[0], alpha, dUz, Uz[1], s);
        Sums S{ctx, s};
        queue_lam24<T>(S, fields());
        queue_lam35<T>(S, m, Au[0], bs, delta);
        set_f(S.fetch());
    }
    void differences() {               // trial - previous, for update_g
        axpy3<T>(n, dU, -1.0, U[1], U[0], s);
        axpy3<T>(n, dg, -1.0, g[1], g[0], s);
        axpy3<T>(n, dg2, -1.0, g2[1], g2[0], s);
        axpy3<T>(m, dAu, -1.0, Au[1], Au[0], s);
        axpy3<T>(n, dUx, -1.0, Ux[1], Ux[0], s);
        axpy3<T>(n, dUy, -1.0, Uy[1], Uy[0], s);
        axpy3<T>(n, dUz, -1.0, Uz[1], Uz[0], s);
    }
    void gradient() { grad<T>(n, d[0], muDbeta, g[0], g2[0], DtsAtd, s); }
    // W, then all that follows from it: update_W (:965-1029), the direction
    // (:896-919), and the sums of the next step length and the stopping test.
    // They go to the next buffers, so they can be queued before the line
    // search of the trial is decided (nearly every trial is accepted; an
    // iteration then waits for the device once).
    void queue_W(Sums &S) {
        queue_shrink<T>(S, next_fields(), iso(), beta);
        queue_next(S);
    }
    void queue_next(Sums &S) {
        queue_update<T>(S, next_fields(), g[0], g[1], g2[1], DtsAtd, U[0], U[1], muDbeta, d[1]);
    }
    PlainFields<T> next_fields() {
        PlainFields<T> F = fields();
        F.Wx = Wx[1]; F.Wy = Wy[1]; F.Wz = Wz[1];
        F.g2 = g2_next;
        return F;
    }
    int iso() const { return o->tv_mode == TV3_TV_ISO; }
    void take_W(const double *v) {
        f -= (lam1 + beta / 2 * lam2 - lam4);
        lam1 = v[0]; lam2 = v[1]; lam4 = v[2];
        dd = v[3]; uu = v[4]; upup = v[5]; ug = v[6];
        f += (lam1 + beta / 2 * lam2 - lam4);
        for (auto *w : {Wx, Wy, Wz, d}) std::swap(w[0], w[1]);
        std::swap(g2[0], g2_next);
    }
    void update_mlp() {
        f += (lam4 + lam5);
        lam4 = mlp_sigma<T>(ctx, n, Ux[0], Uy[0], Uz[0], Wx[0], Wy[0], Wz[0], beta, sx, sy, sz, s);
        lam5 = mlp_delta<T>(ctx, m, Au[0], bs, mu, delta, s);
        f -= (lam4 + lam5);
    }
};

// scaleb (3d/tval3_gpu_3d.cpp:225-266) on a host copy of b: the entries of
// least and largest magnitude, the first on ties.  Magnitudes are compared as
// the integers of their bits, which order alike (a loop the compiler can
// vectorise); the largest tells whether any entry is NaN or Inf.
template <typename T>
double scale_factor_of(const T *b, int64_t m) {
    using I = std::conditional_t<sizeof(T) == 4, int32_t, int64_t>;
    const I mask = std::numeric_limits<I>::max();
    auto bits = [mask](T v) {
        I i;
        std::memcpy(&i, &v, sizeof(T));
        return (I)(i & mask);
    };
    if (m == 0) return 1.0;
    I lo = mask, hi = 0;
    for (int64_t k = 0; k < m; ++k) {
        const I i = bits(b[k]);
        lo = i < lo ? i : lo;
        hi = i > hi ? i : hi;
    }
    TV3_REQUIRE(hi < bits(std::numeric_limits<T>::infinity()), TV3_E_NONFINITE,
                "b holds NaN or Inf");
    auto first = [&](I want) {
        int64_t k = 0;
        while (bits(b[k]) != want) ++k;
        return b[k];
    };
    const T dif = std::fabs(first(hi) - first(lo));
    T s = 1;
    if (dif < (T)0.5) s = (T)0.5 / dif;
    else if (dif > (T)1.5) s = (T)1.5 / dif;
    return (double)s;
}

}  // namespace

template <typename T>
void solve_plain(tv3_ctx *ctx, tv3_op *op, const tv3_opts &o, const int32_t dims[3],
                 const T *b_dev, T *U, const T *Ut_dev, tv3_info *info, tv3_history *hist,
                 const T *b_host) {
    hipStream_t s = ctx->stream;
    PlainState<T> S;
    S.ctx = ctx; S.op = op; S.o = &o; S.s = s;
    for (int a = 0; a < 3; ++a) S.dims[a] = dims[a];
    S.n = (int64_t)dims[0] * dims[1] * dims[2];
    S.m = op->m;
    const int64_t n = S.n, m = S.m;
    S.alloc();

    hipEvent_t ev0, ev1, evl0, evl1;
    TV3_HIP(hipEventCreate(&ev0)); TV3_HIP(hipEventCreate(&ev1));
    TV3_HIP(hipEventCreate(&evl0)); TV3_HIP(hipEventCreate(&evl1));
    TV3_HIP(hipEventRecord(ev0, s));

    // b: scale on the device by the factor found on the host (:1122-1124)
    std::vector<T> bh;
    if (!b_host) {
        bh.resize(m);
        TV3_HIP(hipMemcpyAsync(bh.data(), b_dev, sizeof(T) * m, hipMemcpyDeviceToHost, s));
        TV3_HIP(hipStreamSynchronize(s));
        b_host = bh.data();
    }
    const double scl = scale_factor_of<T>(b_host, m);
    scale<T>(m, S.bs, scl, b_dev, s);

    S.A(true, S.bs, S.Atb);
    if (!o.warm_start) S.copy(S.U[0], S.Atb, n);
    else scale<T>(n, S.U[0], scl, U, s);
    S.mu = std::min(o.mu0, o.mu);
    S.beta = std::min(o.beta0, o.beta);
    S.muDbeta = S.mu / S.beta;
    S.copy(S.rcdU, S.U[0], n);
    launch_D<T>(dims, S.U[0], S.Ux[0], S.Uy[0], S.Uz[0], s);
    {
        Sums L{ctx, s};
        queue_shrink<T>(L, S.fields(), o.tv_mode == TV3_TV_ISO, S.beta);
        S.lam1 = L.fetch()[0];
        S.get_g(L, true, false);
    }
    S.gradient();

    double Q = 1, Qp, C = S.f, gam = o.gam;
    int outer = 0, total = 0, backtracks = 0, fallbacks = 0;
    double RelChg = 0, RelChgOut = 0, nrmup = 0;
    bool nonfinite = false;
    TV3_HIP(hipEventRecord(evl0, s));

    while (outer < o.maxcnt && total < o.maxit) {
        bool fst = true;
        while (total < o.maxit) {
            double tau = fst ? S.first_tau() : std::fabs(S.uu / S.ug);
            S.turn();
            Sums sums{ctx, s};
            const double *next_W = S.descend(sums, tau, false, true);
            double alpha = 1.0;
            const double f_trial = S.f;
            double c_armij = S.dd * tau * o.c * S.beta;
            int cnt = 0;
            if (std::fabs(S.f) > std::fabs(C - alpha * c_armij)) {
                S.differences();
                while (std::fabs(S.f) > std::fabs(C - alpha * c_armij)) {
                    if (cnt == 5) {
                        gam *= o.rate_gam;
                        tau = S.first_tau();
                        S.descend(sums, tau, true, false);
                        cnt = 6;
                        ++fallbacks;
                        break;
                    }
                    alpha *= o.gamma;
                    S.update_g(alpha);
                    ++cnt;
                }
                backtracks += cnt > 5 ? 5 : cnt;
                S.queue_W(sums);           // the queued one was the trial's
                next_W = sums.fetch();
            }
            S.take_W(next_W);
            Qp = Q; Q = gam * Qp + 1; C = (gam * Qp * C + S.f) / Q;
            ++total;
            nrmup = std::sqrt(S.upup);
            RelChg = std::sqrt(S.uu) / nrmup;
            if (hist && hist->count < hist->cap) {
                int k = hist->count++;
                hist->f[k] = S.f; hist->lam1[k] = S.lam1; hist->lam2[k] = S.lam2;
                hist->lam3[k] = S.lam3; hist->lam4[k] = S.lam4; hist->lam5[k] = S.lam5;
                hist->tau[k] = tau; hist->alpha[k] = alpha; hist->relchg[k] = RelChg;
                hist->mu[k] = S.mu; hist->beta[k] = S.beta; hist->C[k] = C;
                hist->cnt[k] = cnt; hist->outer[k] = outer;
                if (hist->mulT) hist->mulT[k] = S.last_mul;
                if (hist->f_trial) hist->f_trial[k] = f_trial;
            }
            if (!std::isfinite(S.f)) { nonfinite = true; break; }
            if (RelChg < o.tol_inn && !fst) break;
            fst = false;
        }
        if (nonfinite) break;
        ++outer;
        auto dn = diff_norm<T>(ctx, n, S.U[0], S.rcdU, s);
        RelChgOut = std::sqrt(dn[0]) / nrmup;
        S.copy(S.rcdU, S.U[0], n);
        if (RelChgOut < o.tol) break;
        S.update_mlp();
        double beta0 = S.beta;
        S.beta *= o.rate_cnt; S.mu *= o.rate_cnt;
        if (S.beta > o.beta) S.beta = o.beta;
        if (S.mu > o.mu) S.mu = o.mu;
        S.muDbeta = S.mu / S.beta;
        S.f = S.fval();
        scale<T>(n, S.DtsAtd, beta0 / S.beta, S.d[0], s);
        S.gradient();
        gam = o.gam; Q = 1; C = S.f;
    }
    TV3_HIP(hipEventRecord(evl1, s));
    divide<T>(n, U, scl, S.U[0], s);    // :1275-1277
    TV3_HIP(hipEventRecord(ev1, s));
    TV3_HIP(hipStreamSynchronize(s));
    float ms = 0, msl = 0;
    TV3_HIP(hipEventElapsedTime(&ms, ev0, ev1));
    TV3_HIP(hipEventElapsedTime(&msl, evl0, evl1));
    info->total_iters = total;
    info->outer_iters = outer;
    info->rel_chg = RelChgOut;
    info->secs = ms / 1000.0;
    info->loop_secs = msl / 1000.0;
    info->backtracks = backtracks;
    info->fallbacks = fallbacks;
    info->n_matvec_N = S.nN;
    info->n_matvec_T = S.nT;
    info->status = nonfinite ? TV3_E_NONFINITE : TV3_OK;
    info->rel_error = 0;
    if (Ut_dev) {
        auto e = diff_norm<T>(ctx, n, Ut_dev, U, s);
        info->rel_error = std::sqrt(e[0]) / std::sqrt(e[1]);
    }
    (void)hipEventDestroy(ev0); (void)hipEventDestroy(ev1);
    (void)hipEventDestroy(evl0); (void)hipEventDestroy(evl1);
}

template void solve_plain<float>(tv3_ctx *, tv3_op *, const tv3_opts &, const int32_t *,
                                 const float *, float *, const float *, tv3_info *, tv3_history *,
                                 const float *);
template void solve_plain<double>(tv3_ctx *, tv3_op *, const tv3_opts &, const int32_t *,
                                  const double *, double *, const double *, tv3_info *,
                                  tv3_history *, const double *);

}  // namespace tv3
