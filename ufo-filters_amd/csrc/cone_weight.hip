// FDK pre-weighting (`cone-beam-projection-weight` task).
//
// out = in * SOD * cos(axis_x) / sqrt(L^2 + x^2 + y^2) with the pixel centre
// (x, y) scaled to the isocentre (conebeam.cl:20-36) and the per-projection
// argument set-up of ufo-cone-beam-projection-weight-task.c:116-158.  One
// launch weights n_proj projections; the scalar arguments of every projection
// are precomputed on the host (FP64 inputs rounded to float like the task).
#include "ufomi_internal.h"

#include <cmath>
#include <vector>

namespace {

struct WeightArgs {
    float cx, cz, sd, overall, mag_recip, cos_angle;
};

constexpr int kProj = 4;  // projections per thread

// A thread weights V adjacent pixels of kProj projections.  Bound by HBM at 8 bytes per pixel: a
// pixel per thread ran at 3.2 TB/s (720 projections of 1024^2: 1.89 ms); here 4 16-byte loads are
// in flight per thread, and the square root is shared while the geometry does not change (1.03 ms,
// 5.8 TB/s).
template <int V>
__global__ __launch_bounds__(256) void cone_weight_kernel(const float *__restrict__ in, float *__restrict__ out,
                                                          int W, int H, int n_proj,
                                                          const WeightArgs *__restrict__ args)
{
    const int i = (blockIdx.x * 64 + (threadIdx.x & 63)) * V;
    const int j = blockIdx.y * 4 + (threadIdx.x >> 6);
    const int p0 = blockIdx.z * kProj;
    if (i >= W || j >= H)
        return;
    using T = typename std::conditional<V == 4, float4, float>::type;
    const long plane = (long) W * H, o = (long) j * W + i;
    T x[kProj];
#pragma unroll
    for (int k = 0; k < kProj; k++)
        if (p0 + k < n_proj) x[k] = *(const T *) (in + (long) (p0 + k) * plane + o);
    float r[V];
    WeightArgs a = {};
#pragma unroll
    for (int k = 0; k < kProj; k++) {
        if (p0 + k >= n_proj) break;
        const WeightArgs b = args[p0 + k];
        if (k == 0 || b.cx != a.cx || b.cz != a.cz || b.overall != a.overall || b.mag_recip != a.mag_recip) {
            const float y = (((float) j) - b.cz + 0.5f) * b.mag_recip;
#pragma unroll
            for (int q = 0; q < V; q++) {
                const float u = (((float) (i + q)) - b.cx + 0.5f) * b.mag_recip;
                r[q] = sqrtf(b.overall * b.overall + u * u + y * y);
            }
        }
        a = b;
        T v = x[k];
        float *f = (float *) &v;
#pragma unroll
        for (int q = 0; q < V; q++) f[q] = f[q] * a.sd * a.cos_angle / r[q];
        *(T *) (out + (long) (p0 + k) * plane + o) = v;
    }
}

double pick(const double *a, int n, int i) { return n == 1 ? a[0] : a[i]; }

}  // namespace

extern "C" int ufomi_cone_weight(ufomi_ctx *ctx, const float *d_in, float *d_out, int W, int H, int n_proj,
                                 const double *center_x, const double *center_z, const double *source_distance,
                                 const double *detector_distance, const double *axis_angle_x, int n_param)
{
    int rc = ufomi_enter(ctx);
    if (rc) return rc;
    if (!d_in || !d_out || W <= 0 || H <= 0 || n_proj <= 0 || n_proj > 65535)
        return ufomi_fail(UFOMI_ERR_ARG, "invalid cone weight arguments");
    if (!center_x || !center_z || !source_distance || !detector_distance || n_param <= 0)
        return ufomi_fail(UFOMI_ERR_ARG, "center-position-x/z, source-distance and detector-distance must be set");
    if (n_param != 1 && n_param < n_proj)
        return ufomi_fail(UFOMI_ERR_ARG, "per-projection arrays need %d values, got %d", n_proj, n_param);

    std::vector<WeightArgs> h(n_proj);
    for (int p = 0; p < n_proj; p++) {
        WeightArgs &a = h[p];
        a.cos_angle = (float) cos(axis_angle_x ? pick(axis_angle_x, n_param, p) : 0.0);
        a.cx = (float) pick(center_x, n_param, p);
        a.cz = (float) pick(center_z, n_param, p);
        a.sd = (float) pick(source_distance, n_param, p);
        const float dd = (float) pick(detector_distance, n_param, p);
        a.overall = a.sd + dd;
        a.mag_recip = a.sd / a.overall;
        if (a.cos_angle > 0.9999999f)
            a.overall = a.sd;
    }
    WeightArgs *d_args = nullptr;
    if ((rc = ufomi_scratch(ctx, n_proj * sizeof(WeightArgs), (void **) &d_args))) return rc;
    if ((rc = ufomi_upload(ctx, d_args, h.data(), n_proj * sizeof(WeightArgs)))) return rc;
    const bool a16 = W % 4 == 0 && (((uintptr_t) d_in | (uintptr_t) d_out) & 15) == 0;
    const int per = a16 ? 256 : 64;
    const dim3 grid((W + per - 1) / per, (H + 3) / 4, (n_proj + kProj - 1) / kProj);
    if (a16)
        hipLaunchKernelGGL(cone_weight_kernel<4>, grid, dim3(256), 0, ctx->stream, d_in, d_out, W, H, n_proj, d_args);
    else
        hipLaunchKernelGGL(cone_weight_kernel<1>, grid, dim3(256), 0, ctx->stream, d_in, d_out, W, H, n_proj, d_args);
    UFOMI_CHECK_LAUNCH();
    return UFOMI_OK;
}
