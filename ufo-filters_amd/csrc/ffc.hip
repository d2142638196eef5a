// Adjacent steps before the reconstruction path:
//  * `flat-field-correct` (src/kernels/ffc.cl:20-48,
//    src/ufo-flat-field-correct-task.c:107-160): per pixel
//      d = dark * dark_scale, f = flat * flat_scale,
//      (data - d) / (f - d), or log((f - d) / (data - d)) with absorption,
//    NaN and Inf replaced by 0 on request; with sinogram input the dark and
//    flat are one row indexed by x.  One launch corrects a batch of items; an
//    item past the last dark (flat) item uses the last one, as a finished
//    input stream keeps feeding its last buffer.
//  * `average` (src/ufo-average-task.c:102-151): the float32 sum of the items
//    in arrival order divided by their count.
// Both are elementwise and bound by HBM.
#include "ufomi_internal.h"

#include <algorithm>

// Every float operation rounds on its own, as in the reference kernels' source
// (hipcc would otherwise fuse a * b + c into one FMA).
#pragma clang fp contract(off)

namespace {

constexpr int kThreads = 256;

// (data - d) / (f - d), or log((f - d) / (data - d)), with f - d given.
__device__ __forceinline__ float ffc_one(float v, float dk, float range, bool absorb, bool fix)
{
    float r = absorb ? logf((range / (v - dk)))
                     : ((v - dk) / range);
    if (fix && (isnan(r) || isinf(r)))
        r = 0.0f;
    return r;
}

constexpr int kItems = 8;  // items per thread, at most

template <int V> struct Vec { float v[V]; };
template <int V> __device__ __forceinline__ Vec<V> load_vec(const float *p)
{
    Vec<V> r;
    if constexpr (V == 4) {
        const float4 q = *(const float4 *) p;
        r.v[0] = q.x; r.v[1] = q.y; r.v[2] = q.z; r.v[3] = q.w;
    } else {
        r.v[0] = *p;
    }
    return r;
}

// A thread corrects V adjacent pixels of kItems items.  Bound by HBM at 8 bytes per pixel: a pixel
// per thread with its own 64-bit division and dark and flat reads ran at 2.5 TB/s (400 items of
// 1024^2: 1.32 ms); here the dark and flat are read once per kItems items while they do not
// change, and 8 16-byte loads are in flight per thread (0.65 ms, 5.1 TB/s).
template <int V>
__global__ __launch_bounds__(kThreads) void ffc_kernel(const float *__restrict__ data, const float *__restrict__ dark,
                                                       const float *__restrict__ flat, float *__restrict__ out,
                                                       long plane, int W, int n, int n_dark, int n_flat,
                                                       int sino_in, int absorb, int fix, float dark_scale,
                                                       float flat_scale, int items)
{
    const long e = ((long) blockIdx.x * kThreads + threadIdx.x) * V;
    if (e >= plane)
        return;
    const long ce = sino_in ? (long) ((unsigned long) e % (unsigned) W) : e;
    const long cplane = sino_in ? W : plane;
    const int i0 = blockIdx.y * items;
    n = min(n, i0 + items);
    Vec<V> x[kItems];
#pragma unroll
    for (int k = 0; k < kItems; k++)
        if (i0 + k < n) x[k] = load_vec<V>(data + (long) (i0 + k) * plane + e);
    Vec<V> dk, range;
#pragma unroll
    for (int k = 0; k < kItems; k++) {
        const int item = i0 + k;
        if (item >= n) break;
        if (k == 0 || item < n_dark || item < n_flat) {
            dk = load_vec<V>(dark + min(item, n_dark - 1) * cplane + ce);
            const Vec<V> fl = load_vec<V>(flat + min(item, n_flat - 1) * cplane + ce);
#pragma unroll
            for (int j = 0; j < V; j++) {
                dk.v[j] = dk.v[j] * dark_scale;
                range.v[j] = fl.v[j] * flat_scale - dk.v[j];
            }
        }
        float r[V];
#pragma unroll
        for (int j = 0; j < V; j++) r[j] = ffc_one(x[k].v[j], dk.v[j], range.v[j], absorb != 0, fix != 0);
        float *o = out + (long) item * plane + e;
        if constexpr (V == 4)
            *(float4 *) o = make_float4(r[0], r[1], r[2], r[3]);
        else
            o[0] = r[0];
    }
}

__global__ __launch_bounds__(kThreads) void average_kernel(const float *__restrict__ in, long elems, int n,
                                                           int copies, float *__restrict__ out)
{
    const long e = (long) blockIdx.x * kThreads + threadIdx.x;
    if (e >= elems)
        return;
    float s = 0.0f;
    for (int k = 0; k < n; k++)
        s = (s + in[(long) k * elems + e]);
    const float m = (s / (float) n);
    for (int c = 0; c < copies; c++)
        out[(long) c * elems + e] = m;
}

}  // namespace

extern "C" int ufomi_flat_field_correct(ufomi_ctx *ctx, const float *d_data, int W, int H, int n,
                                        const float *d_dark, int n_dark, const float *d_flat, int n_flat,
                                        int sinogram_input, int absorption_correct, int fix_nan_and_inf,
                                        float dark_scale, float flat_scale, float *d_out)
{
    int rc = ufomi_enter(ctx);
    if (rc) return rc;
    if (!d_data || !d_dark || !d_flat || !d_out || W <= 0 || H <= 0 || n <= 0 || n_dark <= 0 || n_flat <= 0)
        return ufomi_fail(UFOMI_ERR_ARG, "invalid flat-field arguments");
    const long plane = (long) W * H, total = plane * n;
    if ((total + kThreads - 1) / kThreads >= (1L << 31))
        return ufomi_fail(UFOMI_ERR_ARG, "flat-field batch too large for one launch");
    // 16-byte accesses where every pixel group of an item (and of a dark or flat row) is aligned
    const bool a16 = plane % 4 == 0 && (!sinogram_input || W % 4 == 0) &&
                     (((uintptr_t) d_data | (uintptr_t) d_dark | (uintptr_t) d_flat | (uintptr_t) d_out) & 15) == 0;
    const int per = kThreads * (a16 ? 4 : 1);
    const long bx = (plane + per - 1) / per;
    // fewer items per thread where the grid would not give each of the 256 CUs four workgroups: a
    // thread's items wait for their dark and flat one after the other (2000 rows of 1024 pixels with
    // a dark and a flat each: 9.5 us with 8, 5.0 us with 1)
    int items = kItems;
    while (items > 1 && bx * ((n + items - 1) / items) < 1024) items /= 2;
    // the grid's second axis holds 65535 blocks: longer batches go in several launches
    for (long first = 0; first < n; first += 65535L * items) {
        const int count = (int) std::min<long>(n - first, 65535L * items);
        const dim3 grid((unsigned) bx, (unsigned) ((count + items - 1) / items));
        const long dplane = sinogram_input ? W : plane;
        const float *dk = d_dark + std::min<long>(first, n_dark - 1) * dplane;
        const float *fl = d_flat + std::min<long>(first, n_flat - 1) * dplane;
        const int nd = (int) std::max<long>(1, n_dark - first), nf = (int) std::max<long>(1, n_flat - first);
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, ctx->stream, d_data + first * plane, dk, fl,
                               d_out + first * plane, plane, W, count, nd, nf, sinogram_input, absorption_correct,
                               fix_nan_and_inf, dark_scale, flat_scale, items);
        };
        if (a16) go(ffc_kernel<4>);
        else go(ffc_kernel<1>);
        UFOMI_CHECK_LAUNCH();
    }
    return UFOMI_OK;
}

extern "C" int ufomi_average(ufomi_ctx *ctx, const float *d_items, size_t elems, int n, int copies, float *d_out)
{
    int rc = ufomi_enter(ctx);
    if (rc) return rc;
    if (!d_items || !d_out || !elems || n <= 0 || copies <= 0)
        return ufomi_fail(UFOMI_ERR_ARG, "invalid average arguments");
    const long blocks = ((long) elems + kThreads - 1) / kThreads;
    if (blocks >= (1L << 31))
        return ufomi_fail(UFOMI_ERR_ARG, "average item too large for one launch");
    hipLaunchKernelGGL(average_kernel, dim3((unsigned) blocks), dim3(kThreads), 0, ctx->stream, d_items,
                       (long) elems, n, copies, d_out);
    UFOMI_CHECK_LAUNCH();
    return UFOMI_OK;
}
