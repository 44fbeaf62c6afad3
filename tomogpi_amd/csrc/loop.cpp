// loop.cpp - device-resident simple-gradient reconstruction
// (Iter3D::doSimpleGradient, C/Iter3D_Algo_Gradient.cu:25-223) with the
// generalised-Gaussian beta=2 (quadratic) regulariser
// (C/GeneralizedGaussianRegularizer_CPU.cu:158-226).  Per iteration k:
//   est = P x;  r = y - est;  dJ = B r;  dJ *= -2
//   if lambda != 0:  dJ += (2 lambda) L(L x);
//                    if k < Kopt: normdJProjReg = 2 sum (L dJ)^2
//   if k < Kopt:  est = P dJ;  normdJ = sum dJ^2;
//                 normdJProj = 2 sum est^2 + lambda normdJProjReg
//                 alpha = -normdJ / normdJProj;  alpha_min = max(alpha, alpha_min)
//   else          alpha = alpha_min
//   x += (float)alpha dJ, clamped at 0 if positivity
// With a 16-bit storage type every operator reads a 16-bit copy of its FP32
// input (the mixed-precision form); the rest of the loop is unchanged.
// Volumes, sinograms and the step rule's FP64 norms stay on the device; the
// host takes the statistics at the end.  The SIRT loop (tomo_sirt_run) follows.
#include <algorithm>
#include <cmath>

#include "tomo_internal.hpp"

namespace tomo {
namespace {

struct DevBuf {
    void* p = nullptr;
    ~DevBuf() {
        if (p) (void)hipFree(p);
    }
};

// A loop's work buffer from the stream-ordered pool of the loop's stream,
// released on that stream (after the work queued on it), so allocating and
// releasing it neither waits for the device nor stalls other streams.
struct PoolBuf {
    void* p = nullptr;
    hipStream_t s = nullptr;
    hipError_t alloc(size_t bytes, hipStream_t st) {
        s = st;
        return hipMallocAsync(&p, bytes, st);
    }
    ~PoolBuf() {
        if (p) (void)hipFreeAsync(p, s);
    }
};

// The projector's copy of the volume, allocated once for a loop's run and passed
// to each of its projections (which otherwise take it from the stream-ordered
// pool per call, whose allocations stalled the host for up to seconds now and
// then between the loop's synchronisations).  The compat Siddon reads the volume
// itself and takes none; a Siddon volume beyond its 32-bit traversal index takes
// none either, so that the projector reports it as unsupported.
struct LoopCopies {
    PoolBuf buf;
    ProjExtra extra;
    int alloc(const tomo_geom* g, const tomo_gd_params& pr, int storage, hipStream_t s) {
        const int nx = g->info.nx, ny = g->info.ny, nz = g->info.nz;
        const bool sid = pr.pair == TOMO_PAIR_SIDDONVI;
        if (sid && ((pr.flags & TOMO_FLAG_SIDDON_COMPAT) || !sid_volume_fits(nx, ny, nz))) return TOMO_OK;
        const size_t es = storage == TOMO_F32 ? 4 : 2;
        const int planes = proj_planes(g->dev, !sid && (pr.flags & TOMO_FLAG_RS_FOV_CUBE)).nz;
        TOMO_HIP(buf.alloc(sid ? zcol_words(nx, ny, planes, es) * 4 : rs_copy_shape(nx, ny, planes, es).elems * 8, s));
        extra.copy = buf.p;
        return TOMO_OK;
    }
};

int project(const tomo_geom* g, const tomo_gd_params& pr, const float* vol, float* sino, hipStream_t s,
            const ProjExtra& x) {
    Buf in{vol, TOMO_F32, 1.0f};
    MutBuf out{sino, TOMO_F32, 1.0f};
    if (pr.pair == TOMO_PAIR_SIDDONVI)
        return launch_siddon(g, (pr.flags & TOMO_FLAG_SIDDON_COMPAT) ? 1 : 0, in, out, s, x);
    return launch_rs(g, (pr.flags & TOMO_FLAG_RS_FOV_CUBE) ? 1 : 0, in, out, s, x);
}

// Operator inputs of the mixed-precision loops (tomo_gd_params.storage
// TOMO_F16 / TOMO_BF16): each operator reads a 16-bit copy of its FP32
// input, made in `tmp` (room for the larger of a volume and a sinogram);
// FP16 copies are scaled by the power of two that puts max|x| in
// [2^13, 2^14), BF16 copies are unscaled.  Outputs stay FP32.  The copy is
// reused by the next operator of the same stream, after this one read it.
struct Mixed {
    int dtype = TOMO_F32;
    PoolBuf tmp;
    int init(int storage, size_t n, hipStream_t s) {
        dtype = storage;
        if (dtype != TOMO_F32) TOMO_HIP(tmp.alloc(n * 2, s));
        return TOMO_OK;
    }
    int stage(const float* x, size_t n, Buf* in, hipStream_t s) {
        if (dtype == TOMO_F32) {
            *in = Buf{x, TOMO_F32, 1.0f};
            return TOMO_OK;
        }
        float scale = 1.0f;
        if (dtype == TOMO_F16) {
            float m = 0.0f;
            const int rc = reduce_max_abs(x, n, &m, s);
            if (rc) return rc;
            if (m > 0.0f && std::isfinite(m)) {
                int e = 0;
                (void)std::frexp(m, &e);  // m = f 2^e, f in [0.5, 1)
                scale = std::ldexp(1.0f, std::min(100, std::max(-100, 14 - e)));
            }
        }
        *in = Buf{tmp.p, dtype, scale};
        return launch_convert(Buf{x, TOMO_F32, 1.0f}, MutBuf{tmp.p, dtype, scale}, n, s);
    }
};

int project(const tomo_geom* g, const tomo_gd_params& pr, Mixed& mx, const float* vol, float* sino, hipStream_t s,
            const ProjExtra& x) {
    Buf in{};
    int rc = mx.stage(vol, g->nvox(), &in, s);
    if (rc) return rc;
    const MutBuf out{sino, TOMO_F32, 1.0f};
    if (pr.pair == TOMO_PAIR_SIDDONVI)
        return launch_siddon(g, (pr.flags & TOMO_FLAG_SIDDON_COMPAT) ? 1 : 0, in, out, s, x);
    return launch_rs(g, (pr.flags & TOMO_FLAG_RS_FOV_CUBE) ? 1 : 0, in, out, s, x);
}

int backproject(const tomo_geom* g, Mixed& mx, const float* sino, float* vol, hipStream_t s) {
    Buf in{};
    int rc = mx.stage(sino, g->nsino(), &in, s);
    if (rc) return rc;
    return launch_vi(g, in, MutBuf{vol, TOMO_F32, 1.0f}, s);
}

// The scalars of a loop's run, in device memory: the partial sums of the running
// iteration, the state of the step rule, and the statistics of up to kKept
// iterations, which go to the host when they are full and at the end.  The host
// waits there only: a norm that returned to it after each sum cost about 60 us
// of an idle device, five times an iteration (128^3 and 180 views, 5 iterations:
// 4.53 -> 3.45 ms with the passes fused).
struct LoopScalars {
    static constexpr int kKept = 1024;
    PoolBuf buf;
    LoopStep step{};
    double* partial = nullptr;
    char *stats = nullptr, *host = nullptr;
    size_t entry = 0;
    int kept = 0;
    // iterations: of the run; state: the rule's, initially; host_stats: entries of
    // entry_bytes (a tomo_gd_iter_stat, or its first field alone), or null.
    int alloc(int iterations, double state, void* host_stats, size_t entry_bytes, hipStream_t s) {
        host = (char*)host_stats;
        entry = entry_bytes;
        kept = host ? std::max(1, std::min(iterations, kKept)) : 1;
        const size_t sums = (size_t)kLoopSums * kLoopPartials;
        TOMO_HIP(buf.alloc((sums + 1) * sizeof(double) + kept * sizeof(tomo_gd_iter_stat), s));
        partial = (double*)buf.p;
        stats = (char*)(partial + sums + 1);
        step.partial = partial;
        step.state = partial + sums;
        step.init = state;
        return TOMO_OK;
    }
    double* sum(LoopSum q, size_t n) {
        step.blocks[q] = (int)loop_blocks(n);
        return partial + (size_t)q * kLoopPartials;
    }
    // Begins iteration k (from 0).
    void begin(int k) {
        step.stat = (tomo_gd_iter_stat*)(stats + (size_t)(k % kept) * entry);
        step.first = k == 0;
        step.begins = 1;
    }
    // Ends the sums asked for since the last call.
    int end(LoopRule rule, double lambda, hipStream_t s) {
        step.rule = rule;
        step.lambda = lambda;
        const int rc = launch_loop_step(step, s);
        std::fill(step.blocks, step.blocks + kLoopSums, 0);
        step.begins = 0;
        return rc;
    }
    // After iteration k: the kept statistics to the host when they are full or
    // `last`.  The host is never more than kKept iterations ahead of the device.
    int flush(int k, bool last, hipStream_t s) {
        if (host && (last || (k + 1) % kept == 0)) {
            const int first = k / kept * kept;
            TOMO_HIP(hipMemcpyAsync(host + (size_t)first * entry, stats, (size_t)(k + 1 - first) * entry,
                                    hipMemcpyDeviceToHost, s));
            TOMO_HIP(hipStreamSynchronize(s));
        } else if ((k + 1) % kKept == 0) {
            TOMO_HIP(hipStreamSynchronize(s));
        }
        return TOMO_OK;
    }
};

}  // namespace

int gd_run(tomo_ctx* ctx, const tomo_geom* g, const tomo_gd_params& pr, const float* sino, const float* weight,
           float* vol, tomo_gd_iter_stat* stats, hipStream_t s) {
    (void)ctx;
    const size_t nv = g->nvox(), ns = g->nsino();
    const int nx = g->info.nx, ny = g->info.ny, nz = g->info.nz;
    const bool reg = pr.lambda != 0.0;
    PoolBuf est, dj, t1;
    TOMO_HIP(est.alloc(ns * sizeof(float), s));
    TOMO_HIP(dj.alloc(nv * sizeof(float), s));
    if (reg) TOMO_HIP(t1.alloc(nv * sizeof(float), s));
    Mixed mx;
    int rc = mx.init(pr.storage, std::max(nv, ns), s);
    if (rc) return rc;
    LoopCopies cp;
    if ((rc = cp.alloc(g, pr, pr.storage, s))) return rc;
    LoopScalars sc;
    if ((rc = sc.alloc(pr.gradient_iteration_nb, pr.alpha_min_init, stats, sizeof(*stats), s))) return rc;
    float* e = (float*)est.p;
    float* d = (float*)dj.p;
    float* a = (float*)t1.p;
    for (int k = 1; k <= pr.gradient_iteration_nb; ++k) {
        const bool optimal = k < pr.optimal_step_iteration_nb;
        sc.begin(k - 1);
        if ((rc = project(g, pr, mx, vol, e, s, cp.extra))) return rc;
        // weighted form: r = W (y - P x); the norm is of y - P x
        if ((rc = launch_diff_sq(sino, e, weight, e, ns, sc.sum(kLoopResidual, ns), s))) return rc;
        if ((rc = backproject(g, mx, e, d, s))) return rc;
        if (reg) {
            if ((rc = launch_laplacian_sq(vol, a, nx, ny, nz, sc.sum(kLoopReg, nv), nullptr, s))) return rc;
            const float w = (float)(2.0 * (double)(float)pr.lambda);
            if ((rc = launch_scale_laplacian(a, d, -2.0f, w, nx, ny, nz, s))) return rc;
        } else {
            if ((rc = launch_scale(d, -2.0f, nv, s))) return rc;
        }
        if (optimal) {
            if (reg) {
                double* pd = sc.sum(kLoopDir, nv);
                if ((rc = launch_laplacian_sq(d, nullptr, nx, ny, nz, sc.sum(kLoopDirReg, nv), pd, s))) return rc;
            } else {
                if ((rc = launch_loop_sq(d, nv, sc.sum(kLoopDir, nv), s))) return rc;
            }
            if ((rc = project(g, pr, mx, d, e, s, cp.extra))) return rc;
            if ((rc = launch_loop_sq(e, ns, sc.sum(kLoopProj, ns), s))) return rc;
        }
        if ((rc = sc.end(optimal ? kRuleOptimal : kRuleFixed, pr.lambda, s))) return rc;
        if ((rc = launch_axpy_scalar(vol, d, &sc.step.stat->alpha, pr.positivity, nv, s))) return rc;
        if ((rc = sc.flush(k - 1, k == pr.gradient_iteration_nb, s))) return rc;
    }
    TOMO_HIP(hipStreamSynchronize(s));
    return TOMO_OK;
}

// Conjugate gradient on the criterion of gd_run (Fletcher-Reeves):
//   g = -2 B (y - P x) + 2 lambda L(L x)
//   d = g (k = 1),  d = beta d + g,  beta = |g|^2 / |g_prev|^2
//   alpha = -(g . d) / (2 |P d|^2 + lambda 2 |L d|^2);  x += alpha d
// The reference's doConjugateGradient (C/Iter3D_Algo_Gradient.cu:375-559)
// starts its direction at 0 and divides by that zero norm at iteration 2,
// so this loop defines the method instead of restating it.
int cg_run(tomo_ctx* ctx, const tomo_geom* g, const tomo_gd_params& pr, const float* sino, float* vol,
           tomo_gd_iter_stat* stats, hipStream_t s) {
    (void)ctx;
    const size_t nv = g->nvox(), ns = g->nsino();
    const int nx = g->info.nx, ny = g->info.ny, nz = g->info.nz;
    const bool reg = pr.lambda != 0.0;
    PoolBuf est, gb, db, t1;
    TOMO_HIP(est.alloc(ns * sizeof(float), s));
    TOMO_HIP(gb.alloc(nv * sizeof(float), s));
    TOMO_HIP(db.alloc(nv * sizeof(float), s));
    if (reg) TOMO_HIP(t1.alloc(nv * sizeof(float), s));
    float* e = (float*)est.p;
    float* gr = (float*)gb.p;
    float* d = (float*)db.p;
    float* a = (float*)t1.p;
    Mixed mx;
    int rc = mx.init(pr.storage, std::max(nv, ns), s);
    if (rc) return rc;
    LoopCopies cp;
    if ((rc = cp.alloc(g, pr, pr.storage, s))) return rc;
    LoopScalars sc;
    if ((rc = sc.alloc(pr.gradient_iteration_nb, 0.0, stats, sizeof(*stats), s))) return rc;
    for (int k = 1; k <= pr.gradient_iteration_nb; ++k) {
        sc.begin(k - 1);
        if ((rc = project(g, pr, mx, vol, e, s, cp.extra))) return rc;
        if ((rc = launch_diff_sq(sino, e, nullptr, e, ns, sc.sum(kLoopResidual, ns), s))) return rc;
        if ((rc = backproject(g, mx, e, gr, s))) return rc;
        if (reg) {
            if ((rc = launch_laplacian_sq(vol, a, nx, ny, nz, sc.sum(kLoopReg, nv), nullptr, s))) return rc;
            const float w = (float)(2.0 * (double)(float)pr.lambda);
            if ((rc = launch_scale_laplacian(a, gr, -2.0f, w, nx, ny, nz, s))) return rc;
        } else {
            if ((rc = launch_scale(gr, -2.0f, nv, s))) return rc;
        }
        if ((rc = launch_loop_sq(gr, nv, sc.sum(kLoopDir, nv), s))) return rc;
        if ((rc = sc.end(kRuleBeta, 0.0, s))) return rc;
        if ((rc = launch_direction(gr, d, k == 1 ? nullptr : &sc.step.stat->beta, nv, sc.sum(kLoopDir, nv), s))) return rc;
        if ((rc = project(g, pr, mx, d, e, s, cp.extra))) return rc;
        if ((rc = launch_loop_sq(e, ns, sc.sum(kLoopProj, ns), s))) return rc;
        if (reg) {
            if ((rc = launch_laplacian_sq(d, nullptr, nx, ny, nz, sc.sum(kLoopDirReg, nv), nullptr, s))) return rc;
        }
        if ((rc = sc.end(kRuleConjugate, pr.lambda, s))) return rc;
        if ((rc = launch_axpy_scalar(vol, d, &sc.step.stat->alpha, pr.positivity, nv, s))) return rc;
        if ((rc = sc.flush(k - 1, k == pr.gradient_iteration_nb, s))) return rc;
    }
    TOMO_HIP(hipStreamSynchronize(s));
    return TOMO_OK;
}

// SIRT (defined by this library; the reference has none):
//   R = 1/(P 1), C = relaxation/(B 1), x0 = 0,
//   r = (y - P x) * R;  x = x + C * (B r)  (+ clamp at 0).
int sirt_run(tomo_ctx* ctx, const tomo_geom* g, const tomo_sirt_params& pr, const float* sino, float* vol,
             double* residual_sq, hipStream_t s) {
    (void)ctx;
    const size_t nv = g->nvox(), ns = g->nsino();
    PoolBuf rw, cw, est, b;
    TOMO_HIP(rw.alloc(ns * sizeof(float), s));
    TOMO_HIP(est.alloc(ns * sizeof(float), s));
    TOMO_HIP(cw.alloc(nv * sizeof(float), s));
    TOMO_HIP(b.alloc(nv * sizeof(float), s));
    tomo_gd_params gp{};
    gp.pair = pr.pair;
    gp.flags = pr.flags;
    LoopCopies cp;
    if (const int arc = cp.alloc(g, gp, TOMO_F32, s)) return arc;
    LoopScalars sc;
    if (const int arc = sc.alloc(pr.iterations, 0.0, residual_sq, sizeof(double), s)) return arc;
    float* R = (float*)rw.p;
    float* Cv = (float*)cw.p;
    float* e = (float*)est.p;
    float* bv = (float*)b.p;
    int rc;
    // weights from the operators applied to ones
    if ((rc = launch_fill(bv, 1.0f, nv, s))) return rc;
    if ((rc = project(g, gp, bv, R, s, cp.extra))) return rc;
    if ((rc = launch_recip_weight(R, 1.0f, R, ns, s))) return rc;
    if ((rc = launch_fill(e, 1.0f, ns, s))) return rc;
    if ((rc = launch_vi(g, Buf{e, TOMO_F32, 1.0f}, MutBuf{Cv, TOMO_F32, 1.0f}, s))) return rc;
    if ((rc = launch_recip_weight(Cv, (float)pr.relaxation, Cv, nv, s))) return rc;
    if ((rc = launch_fill(vol, 0.0f, nv, s))) return rc;
    for (int k = 0; k < pr.iterations; ++k) {
        if ((rc = project(g, gp, vol, e, s, cp.extra))) return rc;
        double* part = nullptr;
        if (residual_sq) {
            sc.begin(k);
            part = sc.sum(kLoopResidual, ns);
        }
        if ((rc = launch_diff_sq(sino, e, R, e, ns, part, s))) return rc;
        if (residual_sq && (rc = sc.end(kRuleResidual, 0.0, s))) return rc;
        if ((rc = launch_vi(g, Buf{e, TOMO_F32, 1.0f}, MutBuf{bv, TOMO_F32, 1.0f}, s))) return rc;
        if ((rc = launch_waxpy(vol, Cv, bv, pr.positivity, nv, s))) return rc;
        if ((rc = sc.flush(k, k + 1 == pr.iterations, s))) return rc;
    }
    TOMO_HIP(hipStreamSynchronize(s));
    return TOMO_OK;
}

}  // namespace tomo

extern "C" int tomo_sirt_run(tomo_ctx* ctx, const tomo_geom* g, const tomo_sirt_params* params,
                             const float* sinogram, float* volume, double* residual_sq, void* stream) {
    using namespace tomo;
    if (!ctx || !g || !params || !sinogram || !volume) return fail(TOMO_ERR_INVALID_ARG, "null argument");
    TOMO_HIP(hipSetDevice(ctx->device));
    if (params->pair != TOMO_PAIR_RSVI && params->pair != TOMO_PAIR_SIDDONVI)
        return fail(TOMO_ERR_INVALID_ARG, "unknown pair");
    if (params->iterations < 0) return fail(TOMO_ERR_INVALID_ARG, "negative iteration count");
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (!(params->flags & TOMO_FLAG_HOST_PTR)) return sirt_run(ctx, g, *params, sinogram, volume, residual_sq, s);
    const size_t nv = g->nvox(), ns = g->nsino();
    DevBuf ds, dv;
    TOMO_HIP(hipMalloc(&ds.p, ns * sizeof(float)));
    TOMO_HIP(hipMalloc(&dv.p, nv * sizeof(float)));
    TOMO_HIP(hipMemcpyAsync(ds.p, sinogram, ns * sizeof(float), hipMemcpyHostToDevice, s));
    int rc = sirt_run(ctx, g, *params, (const float*)ds.p, (float*)dv.p, residual_sq, s);
    if (rc) return rc;
    TOMO_HIP(hipMemcpyAsync(volume, dv.p, nv * sizeof(float), hipMemcpyDeviceToHost, s));
    TOMO_HIP(hipStreamSynchronize(s));
    return TOMO_OK;
}

namespace {
// Shared entry of tomo_gd_run / tomo_cg_run: argument checks and host staging.
template <typename Run>
int run_loop(tomo_ctx* ctx, const tomo_geom* g, const tomo_gd_params* params, const float* sinogram, float* volume,
             tomo_gd_iter_stat* stats, void* stream, Run run) {
    using namespace tomo;
    if (!ctx || !g || !params || !sinogram || !volume) return fail(TOMO_ERR_INVALID_ARG, "null argument");
    TOMO_HIP(hipSetDevice(ctx->device));
    if (params->pair != TOMO_PAIR_RSVI && params->pair != TOMO_PAIR_SIDDONVI)
        return fail(TOMO_ERR_INVALID_ARG, "unknown pair");
    if (params->gradient_iteration_nb < 0) return fail(TOMO_ERR_INVALID_ARG, "negative iteration count");
    if (params->storage != TOMO_F32 && params->storage != TOMO_F16 && params->storage != TOMO_BF16)
        return fail(TOMO_ERR_INVALID_ARG, "storage must be TOMO_F32, TOMO_F16 or TOMO_BF16");
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (!(params->flags & TOMO_FLAG_HOST_PTR)) return run(ctx, g, *params, sinogram, volume, stats, s);
    const size_t nv = g->nvox(), ns = g->nsino();
    DevBuf ds, dv;
    TOMO_HIP(hipMalloc(&ds.p, ns * sizeof(float)));
    TOMO_HIP(hipMalloc(&dv.p, nv * sizeof(float)));
    TOMO_HIP(hipMemcpyAsync(ds.p, sinogram, ns * sizeof(float), hipMemcpyHostToDevice, s));
    TOMO_HIP(hipMemcpyAsync(dv.p, volume, nv * sizeof(float), hipMemcpyHostToDevice, s));
    int rc = run(ctx, g, *params, (const float*)ds.p, (float*)dv.p, stats, s);
    if (rc) return rc;
    TOMO_HIP(hipMemcpyAsync(volume, dv.p, nv * sizeof(float), hipMemcpyDeviceToHost, s));
    TOMO_HIP(hipStreamSynchronize(s));
    return TOMO_OK;
}
}  // namespace

extern "C" int tomo_cg_run(tomo_ctx* ctx, const tomo_geom* g, const tomo_gd_params* params, const float* sinogram,
                           float* volume, tomo_gd_iter_stat* stats, void* stream) {
    return run_loop(ctx, g, params, sinogram, volume, stats, stream, tomo::cg_run);
}

extern "C" int tomo_gd_run(tomo_ctx* ctx, const tomo_geom* g, const tomo_gd_params* params, const float* sinogram,
                           float* volume, tomo_gd_iter_stat* stats, void* stream) {
    return run_loop(ctx, g, params, sinogram, volume, stats, stream,
                    [](tomo_ctx* c, const tomo_geom* gg, const tomo_gd_params& pr, const float* y, float* x,
                       tomo_gd_iter_stat* st, hipStream_t s) { return tomo::gd_run(c, gg, pr, y, nullptr, x, st, s); });
}

extern "C" int tomo_wgd_run(tomo_ctx* ctx, const tomo_geom* g, const tomo_gd_params* params, const float* sinogram,
                            const float* weight, float* volume, tomo_gd_iter_stat* stats, void* stream) {
    using namespace tomo;
    if (!weight) return fail(TOMO_ERR_INVALID_ARG, "null weight sinogram");
    DevBuf dw;
    const float* w = weight;
    if (ctx && g && params && (params->flags & TOMO_FLAG_HOST_PTR)) {
        TOMO_HIP(hipSetDevice(ctx->device));
        const size_t ns = g->nsino();
        TOMO_HIP(hipMalloc(&dw.p, ns * sizeof(float)));
        TOMO_HIP(hipMemcpy(dw.p, weight, ns * sizeof(float), hipMemcpyHostToDevice));
        w = (const float*)dw.p;
    }
    return run_loop(ctx, g, params, sinogram, volume, stats, stream,
                    [w](tomo_ctx* c, const tomo_geom* gg, const tomo_gd_params& pr, const float* y, float* x,
                        tomo_gd_iter_stat* st, hipStream_t s) { return gd_run(c, gg, pr, y, w, x, st, s); });
}
