// Gradient-domain phase-contrast reconstruction (IR::gradReconstruct,
// reconstruct.cu:158-328) and its Poisson integration (poissonSolveLDLT,
// poisson_cpu.cpp:15-112) behind the C ABI.
//
// The gradient slots reuse the projector kernels through an XR_CONV_GRAD plan
// of side N+1: the same voxel-driven splat / gather, with the source on the
// -y side, the half-voxel-shifted grid and a constant vox_size in place of the
// chord normalisation.  Slots run one after another; each is an OS-ART (or
// OS-EM) solve like xr_ir_reconstruct's, with the subset order of a fresh
// default-seeded mt19937_64, which is the order the reference's single engine
// gives every slot (it shuffles once per epoch for all of them).
#include <algorithm>
#include <cmath>
#include <memory>
#include <random>
#include <vector>

#include "xr_host.hpp"

using namespace xr;
using namespace xr::host;

namespace {

// subset s holds views (s + batch*j) % P, j < ceil(P/batch) (reconstruct.cu:240-242)
void subset_views(int sub, int batch, int P, std::vector<int>& out) {
    const int ss = (P + batch - 1) / batch;
    out.resize(ss);
    for (int j = 0; j < ss; j++) out[j] = (sub + batch * j) % P;
}

// Workspace of xr_poisson_solve that a context keeps: 512^3 in one piece.
constexpr int64_t kPoissonBytes = 1200ll << 20;

}  // namespace

int xr_poisson_solve(xr_context* ctx, int n, const float* gx, const float* gy, float* vol) {
    if (!ctx || !gx || !gy || !vol) return fail(ctx, XR_ERR_INVALID, "bad args");
    if (n < 3 || n > 4096) return fail(ctx, XR_ERR_INVALID, "poisson solve needs 3 <= n <= 4096 (got %d)", n);
    const int64_t M = n - 2, He = (M + 1) / 2, Ho = M / 2;
    // Tables, then the modes of as many slices as fit the workspace.  The
    // context keeps the buffer (allocating and freeing a gigabyte costs as much
    // as a solve): at most kPoissonBytes, or one slice where that is larger.
    const int64_t tables = He * He + He * Ho + M * M;
    const int64_t slices = std::max<int64_t>(1, std::min<int64_t>(n, (kPoissonBytes / 8 - tables) / (M * M)));
    const size_t need = (size_t)(tables + slices * M * M);
    if (ctx->poisson_len < need) {
        if (ctx->d_poisson) (void)hipFree(ctx->d_poisson);
        ctx->d_poisson = nullptr;
        ctx->poisson_len = 0;
        XR_HIP(ctx, device_malloc((void**)&ctx->d_poisson, need * sizeof(double)));
        ctx->poisson_len = need;
    }
    double* const Se = ctx->d_poisson;
    double* const So = Se + He * He;
    double* const G = So + He * Ho;
    double* const T = G + M * M;
    XR_TRY(timed(ctx, 3, [&] { return launch_poisson_tables(Se, So, G, n, ctx->stream); }));
    XR_TRY(timed(ctx, 3, [&] { return launch_poisson_border(vol, n, ctx->stream); }));
    for (int64_t z0 = 0; z0 < n; z0 += slices)
        XR_TRY(timed(ctx, 3, [&] {
            return launch_poisson_slices(gx, gy, Se, So, G, T, vol, n, (int)z0, (int)std::min<int64_t>(slices, n - z0),
                                         ctx->stream);
        }));
    // the next call, perhaps on another stream, overwrites the workspace
    XR_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return XR_OK;
}

int xr_grad_reconstruct(xr_context* ctx, const xr_geometry* g, const xr_scan* s, const float* sino, float* vol,
                        float* const* grad, int epochs, int batch, int direction, int method, float lambda,
                        int block_size, xr_stats* stats) {
    if (!ctx) return XR_ERR_INVALID;
    XR_TRY(check_geometry(ctx, g));
    XR_TRY(check_scan(ctx, s));
    if (!sino || !vol) return fail(ctx, XR_ERR_INVALID, "sinogram / volume missing");
    if (g->n_vox < 3) return fail(ctx, XR_ERR_INVALID, "gradient reconstruction needs N >= 3");
    if (epochs < 0 || batch <= 0 || batch > g->n_proj) return fail(ctx, XR_ERR_INVALID, "bad epochs / batch");
    if (method != XR_METHOD_MLEM && method != XR_METHOD_ART) return fail(ctx, XR_ERR_INVALID, "method must be MLEM or ART");
    if (block_size <= 0) return fail(ctx, XR_ERR_INVALID, "block_size must be positive");
    const int N = g->n_vox, N1 = N + 1, P = g->n_proj, C = s->n_cond;
    xr_geometry g1 = *g;
    g1.n_vox = N1;  // geom.voxel + 1 (reconstruct.cu:161)
    xr_plan* plan = nullptr;
    XR_TRY(xr_plan_create(ctx, &g1, s, XR_CONV_GRAD, direction, &plan));
    std::unique_ptr<xr_plan, void (*)(xr_plan*)> guard(plan, xr_plan_destroy);
    const int ext = (int)std::min<int64_t>(N1, ((int64_t)N + block_size - 1) / block_size * block_size);
    // the layers z >= ext are held at zero while projecting: no projector pass
    // visits them, the weight pass of the plan's tables included (a 513-voxel
    // column is then 8 chunks of 64, not 9)
    plan->dims.nz = ext;
    XR_TRY(ensure_norm(plan));
    const int64_t V1 = (int64_t)N1 * N1 * N1, lenP = (int64_t)g->n_det_u * g->n_det_v, lenD = lenP * P;
    const int ss = (P + batch - 1) / batch;
    const size_t per_epoch = (size_t)batch * ss;
    DevBuf<float> dref, dvol, dsino0, dsino, dproj, dcoef, dgx, dgy, dout;
    DevBuf<int32_t> dcodes;
    DevBuf<uint8_t> dflags;
    XR_HIP(ctx, dref.alloc(V1));
    XR_HIP(ctx, dvol.alloc(V1));
    XR_HIP(ctx, dsino0.alloc(lenD));
    XR_HIP(ctx, dsino.alloc(lenD));
    XR_HIP(ctx, dproj.alloc(lenD));
    SolveSums sums;
    XR_HIP(ctx, sums.alloc(epochs, batch));
    XR_HIP(ctx, dcoef.alloc(P));
    XR_HIP(ctx, dgx.alloc(V1));
    XR_HIP(ctx, dgy.alloc(V1));
    XR_HIP(ctx, dout.alloc((int64_t)N * N * N));
    XR_HIP(ctx, dcodes.alloc(per_epoch * std::max(epochs, 1)));
    XR_HIP(ctx, dflags.alloc(per_epoch * std::max(epochs, 1)));
    XR_HIP(ctx, hipMemcpyAsync(dsino0.p, sino, sizeof(float) * lenD, hipMemcpyHostToDevice, ctx->stream));
    const float alpha = (method == XR_METHOD_ART) ? lambda / (float)ss : 0.f;
    const int kind = (method == XR_METHOD_MLEM) ? BWD_MLEM : BWD_ART;
    const int out_mode = (method == XR_METHOD_MLEM) ? OUT_RATIO : OUT_RESIDUAL;
    std::vector<int32_t> codes(per_epoch * std::max(epochs, 1));
    std::vector<uint8_t> flags(codes.size());
    std::vector<float> coef(P);
    std::vector<int> sv;
    for (int c = 0; c < C; c++) {
        // the subset order every slot sees; views repeated within an epoch
        // accumulate onto their image (proj is zeroed once per epoch, :231)
        std::vector<int> order(batch);
        for (int i = 0; i < batch; i++) order[i] = i;
        std::mt19937_64 rng;
        for (int ep = 0; ep < epochs; ep++) {
            std::shuffle(order.begin(), order.end(), rng);
            std::vector<char> visited(P, 0);
            for (int pos = 0; pos < batch; pos++) {
                subset_views(order[pos], batch, P, sv);
                for (int j = 0; j < ss; j++) {
                    const size_t i = (size_t)ep * per_epoch + (size_t)pos * ss + j;
                    codes[i] = c * P + sv[j];
                    flags[i] = visited[sv[j]];
                    visited[sv[j]] = 1;
                }
            }
        }
        if (epochs > 0) {
            XR_HIP(ctx, hipMemcpyAsync(dcodes.p, codes.data(), codes.size() * sizeof(int32_t), hipMemcpyHostToDevice,
                                       ctx->stream));
            XR_HIP(ctx, hipMemcpyAsync(dflags.p, flags.data(), flags.size(), hipMemcpyHostToDevice, ctx->stream));
        }
        for (int d = 0; d < 3; d++) {
            const int slot = 3 * c + d;
            // sinogramGradientCoef: {cos, sin, 1}[d] of the FP32 angle of view n >= 0
            for (int n = 0; n < P; n++) {
                const double th = (double)theta_f32(n, P);
                coef[n] = d == 0 ? (float)std::cos(th) : d == 1 ? (float)std::sin(th) : 1.0f;
            }
            XR_HIP(ctx, hipMemcpyAsync(dcoef.p, coef.data(), sizeof(float) * P, hipMemcpyHostToDevice, ctx->stream));
            XR_TRY(timed(ctx, 3, [&] { return launch_scale_views(dsino0.p, dsino.p, dcoef.p, lenP, P, ctx->stream); }));
            // 0.01 everywhere (:168); the layers outside the launches are held
            // at zero while projecting and get their 0.01 back at the end
            XR_HIP(ctx, launch_fill(dvol.p, V1, 0.01f, ctx->stream));
            XR_HIP(ctx, launch_grad_faces(dvol.p, N1, ext, 0.0f, ctx->stream));
            XR_HIP(ctx, sums.clear(ctx->stream));
            for (int ep = 0; ep < epochs; ep++)
                for (int pos = 0; pos < batch; pos++) {
                    const size_t off = (size_t)ep * per_epoch + (size_t)pos * ss;
                    float* const vmax = sums.vmax(ep, pos);
                    XR_TRY(forward_launch(plan, FWD_PLAIN, dvol.p, 0, dproj.p, dsino.p, c * P, dcodes.p + off,
                                          dflags.p + off, ss, out_mode, sums.loss(ep), ep + pos ? vmax - 1 : nullptr));
                    XR_TRY(backward_launch(plan, kind, dproj.p, c * P, dcodes.p + off, ss, dvol.p, nullptr, nullptr,
                                           alpha, 0, reinterpret_cast<unsigned*>(vmax)));
                    // the update touched the skipped layers too: back to zero (the
                    // max left in vmax may count them, a bound that stays safe)
                    XR_HIP(ctx, launch_grad_faces(dvol.p, N1, ext, 0.0f, ctx->stream));
                }
            if (stats && stats->losses && epochs > 0)
                XR_HIP(ctx, hipMemcpyAsync(&stats->losses[(size_t)slot * epochs], sums.loss(0),
                                           sizeof(double) * epochs, hipMemcpyDeviceToHost, ctx->stream));
            XR_HIP(ctx, launch_grad_faces(dvol.p, N1, ext, 0.01f, ctx->stream));
            float* dst = (c == 0 && d == 0) ? dgx.p : (c == 0 && d == 1) ? dgy.p : dref.p;
            XR_TRY(xr_volume_from_columns(ctx, dvol.p, dst, N1, 1));
            if (grad && grad[slot])
                XR_HIP(ctx, hipMemcpyAsync(grad[slot], dst, sizeof(float) * V1, hipMemcpyDeviceToHost, ctx->stream));
        }
    }
    XR_TRY(xr_poisson_solve(ctx, N, dgx.p, dgy.p, dout.p));
    XR_HIP(ctx, hipMemcpyAsync(vol, dout.p, sizeof(float) * N * N * N, hipMemcpyDeviceToHost, ctx->stream));
    XR_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return XR_OK;
}
