// Parallel-beam backprojection of stacks of slices on the matrix cores.
//
// The slices of a stack share their geometry, so at one angle the linear
// interpolation of a block of 16 voxels is a small matrix product:
//     acc[voxel][slice] += sum_j w[voxel][j] sino[j][slice]
// with w the hat weights (1 - f, f) of each voxel over the block's detector
// window.  A 4 x 4 block spans at most 3 sqrt 2 = 4.25 detector pixels at any
// angle, so its window is 8 entries, and v_mfma_f32_16x16x32_f16 contracts
// four angles (K = 4 x 8) for 16 voxels and 16 slices: 1024 updates in 16
// matrix cycles.
//
// f16 operands keep float32 results by splitting: a sample, scaled per slice
// by a power of two to below 2^15, is h + l with h, l in f16 (22 bits, and an
// absolute floor of 2^-40 of the slice's maximum); a weight is a multiple of
// 2^-11 plus a remainder of at most 2^-12 in f16 (to 2^-24).  Three products
// (l w_h, h w_l, h w_h) leave out only l w_l, 2^-23 of the term.  f16 storage
// needs no l plane and two products; bf16 storage likewise (8 significant bits
// down to 2^-32 of the slice's maximum).
//
// The floor is absolute, so one large sample would take the precision of its
// whole slice.  A slice of which more than 1 / 64 of the non-zero samples lie
// below kSmall, or 1 / 1024 a further 2^-5 below (a voxel near the axis meets a
// few columns only), is left to the interpolating kernel with its unit, as is one
// that holds an Inf or a NaN.  At kSmall the floor is 2^-18 (4e-6) of a sample in
// f32 storage; half a slice of noise free samples can lie between that and the full
// 22 bits (2^-17 of the maximum) where a small object's filtered rows fall off,
// 6e-3 of it below and 2e-4 of it 2^-5 further.  Noise puts 1e-6 of the samples there.
#include "ufomi_internal.h"

#include <algorithm>
#include <cmath>

namespace {

constexpr int kTile = 32;    // voxels per tile side
constexpr int kSpan = 48;    // staged detector entries per angle: floor(31 sqrt 2 - 3 sqrt 2 + 1) + 8
constexpr int kPad = 48;     // zero entries on both sides of a stored row
constexpr int kSub = 32;     // slices per stored row
constexpr int kRow = kSub * 2;             // bytes of one plane's row of one detector entry
constexpr int kPlane = kSpan * kRow;       // bytes of one staged plane of one angle
constexpr int kParChunk = 64;              // angles per parameter chunk
// Scaled samples below this, 2^-21 of the slice's maximum in f32 storage, keep fewer than 18 bits; in
// bf16 fewer than their 8; f16 ones are exact.
template <typename T> constexpr float kSmall = 0x1p-7f;
template <> constexpr float kSmall<__hip_bfloat16> = 0x1p-17f;
template <> constexpr float kSmall<__half> = 0.0f;
constexpr unsigned kSmallShare = 64, kTinyWeight = 16;  // samples below kSmall / 32 count 16 times
constexpr unsigned kLeftOut = 0x7f800000u;  // from here on, a slice's word of maxbits leaves its unit out
constexpr int kGridY = 65535;  // a grid's second axis: the angles of split_kernel, the slices of absmax_kernel
// Row workspace of a call: as many groups as fit, one at least; a larger group takes the other path.
// Partial volumes (fewer than 2048 workgroups' of 256 KiB) come on top.
constexpr size_t kWorkspace = (size_t) 1 << 30, kGroupMax = (size_t) 4 << 30;

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef unsigned uint4_t __attribute__((ext_vector_type(4)));
typedef __fp16 fp16x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float to_float(float v) { return v; }
__device__ __forceinline__ float to_float(__half v) { return __half2float(v); }
__device__ __forceinline__ float to_float(__hip_bfloat16 v) { return __bfloat162float(v); }

__global__ __launch_bounds__(256) void clear_kernel(unsigned *__restrict__ p, int n)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0;
}

// Largest |v| of every slice, as the bits of a float: ordered like the value, Inf and NaN above all.
// Also the number of its non-zero samples.
template <typename T>
__global__ __launch_bounds__(256) void absmax_kernel(const T *__restrict__ sino, long pitch, long n,
                                                     unsigned *__restrict__ maxbits, unsigned *__restrict__ nonzero)
{
    const T *s = sino + (long) blockIdx.y * pitch;
    const long step = (long) gridDim.x * 256;
    unsigned m = 0, c = 0;
    auto add = [&](T v) {
        const unsigned bits = __float_as_uint(to_float(v)) & 0x7fffffffu;
        m = max(m, bits);
        c += bits != 0;
    };
    long i = (long) blockIdx.x * 256 + threadIdx.x;
    for (; i + 7 * step < n; i += 8 * step) {
        T v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = s[i + k * step];
#pragma unroll
        for (int k = 0; k < 8; k++) add(v[k]);
    }
    for (; i < n; i += step) add(s[i]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        m = max(m, (unsigned) __shfl_xor((int) m, o, 64));
        c += (unsigned) __shfl_xor((int) c, o, 64);
    }
    __shared__ unsigned red[4], cnt[4];
    if ((threadIdx.x & 63) == 0) {
        red[threadIdx.x >> 6] = m;
        cnt[threadIdx.x >> 6] = c;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        atomicMax(maxbits + blockIdx.y, max(max(red[0], red[1]), max(red[2], red[3])));
        atomicAdd(nonzero + blockIdx.y, cnt[0] + cnt[1] + cnt[2] + cnt[3]);
    }
}

// Power of two that takes the slice's maximum into [2^14, 2^15), or for one plane, whose samples
// have at most 11 bits, into [2^15, 2^16): f16 storage is never scaled down, and so exact.
template <int PL> __device__ __forceinline__ int scale_exponent(unsigned maxbits)
{
    if (maxbits == 0 || maxbits >= kLeftOut) return 0;
    return min(16 - PL + 127 - (int) (maxbits >> 23), 126);
}

// Scaled and split rows, slices innermost: ws[group][angle][plane][detector entry][32 slices] f16,
// kPad zero entries on both sides, zero rows up to a multiple of 4 angles.  The two halves of a
// row swap places at odd angles (the bank layout of the tile kernel's reads).  Counts the small
// samples of a slice and marks it in maxbits when they are too many; what its rows hold from then
// on is not used.
template <typename T, int PL>
__global__ __launch_bounds__(256) void split_kernel(const T *__restrict__ sino, long pitch, int W, int P, int Wp,
                                                    int n_slices, unsigned *maxbits,
                                                    const unsigned *__restrict__ nonzero, unsigned *small,
                                                    uint4_t *__restrict__ ws, long group_stride)
{
    constexpr int PITCH = kSub / 2 + 1;  // dwords per entry in LDS
    __shared__ unsigned tile[PL][64 * PITCH];
    const int e0 = blockIdx.x * 64, p = blockIdx.y, g = blockIdx.z;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int j = e0 + lane - kPad;
    const bool in = p < P && j >= 0 && j < W;
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int s = g * kSub + wv * 8 + k;
        v[k] = in && s < n_slices ? to_float(sino[(long) s * pitch + (long) p * W + j]) : 0.0f;
    }
    unsigned few = 0;  // small samples of slice wv * 8 + lane, lane < 8, the smallest ones weighted
#pragma unroll
    for (int k = 0; k < 8; k += 2) {
        unsigned hp = 0, lp = 0;
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int s = g * kSub + wv * 8 + k + q;
            const float x = ldexpf(v[k + q], scale_exponent<PL>(maxbits[min(s, n_slices - 1)]));
            if constexpr (kSmall<T> > 0.0f) {
                const bool some = v[k + q] != 0.0f;
                const unsigned c = __popcll(__ballot(some && fabsf(x) < kSmall<T>));
                const unsigned c2 = __popcll(__ballot(some && fabsf(x) < kSmall<T> / 32));
                if (lane == k + q) few = c + (kTinyWeight - 1) * c2;
            }
            const _Float16 h = (_Float16) x;
            hp |= (unsigned) __builtin_bit_cast(unsigned short, h) << (16 * q);
            if constexpr (PL == 2) {
                const _Float16 l = (_Float16) (x - (float) h);
                lp |= (unsigned) __builtin_bit_cast(unsigned short, l) << (16 * q);
            }
        }
        tile[0][lane * PITCH + wv * 4 + k / 2] = hp;
        if constexpr (PL == 2) tile[PL - 1][lane * PITCH + wv * 4 + k / 2] = lp;
    }
    if constexpr (kSmall<T> > 0.0f) {
        // a slice that is marked already (read past the caches) is not counted on: its counter
        // would be all that the waves wait for
        const int s = g * kSub + wv * 8 + lane;  // < n_slices where few > 0: the padding is zeros
        if (few && __hip_atomic_load(maxbits + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < kLeftOut) {
            const unsigned limit = nonzero[s] / kSmallShare, before = atomicAdd(small + s, few);
            if (before <= limit && before + few > limit) atomicMax(maxbits + s, kLeftOut);
        }
    }
    __syncthreads();
    const int e = threadIdx.x >> 2, part = threadIdx.x & 3;
    if (e0 + e >= Wp) return;
    uint4_t *dst = ws + (long) g * group_stride;
#pragma unroll
    for (int pl = 0; pl < PL; pl++) {
        const unsigned *t = &tile[pl][e * PITCH + part * 4];
        dst[(((long) p * PL + pl) * Wp + e0 + e) * 4 + (part ^ ((p & 1) << 1))] = uint4_t{t[0], t[1], t[2], t[3]};
    }
}

// Lane `B` of each row of 16 lanes, in every lane of the row (DPP row_newbcast).  Used as an
// addend only: folded into a reversed subtraction, the broadcast reached the other operand.
template <int B> __device__ __forceinline__ int row_bcast(int v)
{
    return __builtin_amdgcn_mov_dpp(v, 0x150 + B, 0xf, 0xf, true);
}

// f16 pair (e, f) - h for the f16 pair h: one fused conversion each.
__device__ __forceinline__ unsigned residue(unsigned h, float e, float f)
{
    unsigned l;
    asm("v_fma_mixlo_f16 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(l) : "v"(h), "v"(e));
    asm("v_fma_mixhi_f16 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(l) : "v"(h), "v"(f));
    return l;
}

template <int I, int N, typename F> __device__ __forceinline__ void static_for(F &&f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>());
        static_for<I + 1, N>(f);
    }
}

using LdsShort4 = __attribute__((address_space(3))) short4_t;
using LdsUint4 = __attribute__((address_space(3))) uint4_t;
using LdsChar = __attribute__((address_space(3))) char;

// Entries j .. j + 3 of this lane's slice column, from the 4 x 16 f16 tile the 16 lanes address.
__device__ __forceinline__ short4_t read_tr(const LdsChar *p)
{
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsShort4 *) p);
}

// 16 bytes per lane from src (uniform) + offset to LDS address dst (uniform) + 16 lane, in flight
// until the caller's vmcnt wait.  Written out because the compiler, which cannot tell the two
// staging buffers apart, waits for the builtin's loads before the next LDS read (64 slices of
// 720 x 2048: 8.6 ms with that wait, 7.4 without).  Nothing else here uses m0 (a reserved
// register, so not to be declared).
__device__ __forceinline__ void load_lds(unsigned dst, const char *src, unsigned offset)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(dst), "v"(offset), "s"(src)
                 : "memory");
}

__device__ __forceinline__ int xcd_remap(int b, int nb)
{
    const int q = nb >> 3;
    if (b < (q << 3))
        return (b & 7) * q + (b >> 3);
    return b;
}

// NG row groups of 32 slices per workgroup, NT 16-slice tiles of each group, PL planes, NW waves.
// 128 accumulators per lane (64 with NT = 1): two (three) waves per SIMD.
template <int NG, int NT, int PL, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NT == 1 ? 3 : 2))) void bp_mfma_kernel(
    const char *__restrict__ ws, long group_bytes, int Wp, int W, int P, const float2 *__restrict__ trig, float axis,
    float roi_x, float roi_y, int roi_w, int roi_h, int n_slices, const unsigned *__restrict__ maxbits,
    float *__restrict__ out, long out_pitch, long part_pitch, int tiles_x, int tiles_y, int p_chunk, int p_norm)
{
    constexpr int UNIT = NG * NT * 16;            // slices per workgroup
    constexpr int BPW = 64 / NW;                  // 4 x 4 voxel blocks per wave
    constexpr int QUAD = 4 * NG * PL * kPlane;    // staged bytes of four angles
    constexpr int LOADS = QUAD / 1024 / NW;       // 16-byte loads per lane and quad
    static_assert(QUAD % (1024 * NW) == 0, "whole wave loads");
    __shared__ __align__(64) char buf[2][QUAD];
    __shared__ float4 par[2][kParChunk];          // (sin, cos, offset, stored row)
    __shared__ uint4_t seltab[8];

    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tiles = tiles_x * tiles_y;
    const int nb = tiles * ((n_slices + UNIT - 1) / UNIT);
    const int b = xcd_remap(blockIdx.x, nb);
    const int unit = b / tiles;
    // tiles in columns of a band of 8 rows: the 32 tiles an XCD runs at a time are 8 x 4, whose
    // detector windows overlap most
    const int band = b % tiles / (8 * tiles_x), in_band = b % tiles - band * 8 * tiles_x;
    const int band_h = min(8, tiles_y - 8 * band);
    const int ty = 8 * band + in_band % band_h, tx = in_band / band_h;
    const int slice0 = unit * UNIT;
    // a slice that holds an Inf or a NaN would spread it over a block, and one of too many small
    // samples would lose them: such a unit is left to the interpolating kernel, which runs after
    // this one
    if (__ballot(maxbits[min(slice0 + min(lane, UNIT - 1), n_slices - 1)] >= kLeftOut)) return;
    const int p0 = (int) blockIdx.y * p_chunk;
    const int np = min(p_chunk, P - p0);
    const int nq = (np + 3) >> 2;
    const char *base = ws + (long) unit * NG * group_bytes;
    const int x0 = tx * kTile, y0 = ty * kTile;
    // voxel (0, 0) of the tile, as backproject.cl:63-64 writes a voxel's coordinates
    const float bx0 = (float) x0 - axis + roi_x + 0.5f, by0 = (float) y0 - axis + roi_y + 0.5f;

    if (tid < 8) {
        uint4_t s;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int t = tid - 2 * k;
            s[k] = t == 0 ? 0x03020100u : t == 1 ? 0x01000c0cu : t == -1 ? 0x0c0c0302u : 0x0c0c0c0cu;
        }
        seltab[tid] = s;
    }
    // The detector position of the tile's voxel (0, 0) relative to the staged window's first
    // entry, formed in FP64: what remains is below 48 and keeps 2^-19 in float.
    auto parameters = [&](int chunk) {
        if (tid < kParChunk) {
            const int p = p0 + chunk * kParChunk + tid;
            const float2 sc = trig[min(p, P - 1)];
            const double s = sc.x, c = sc.y;
            const double u0 = (double) bx0 * c + (double) by0 * s + ((double) axis - 0.5);
            const double lo = floor(u0 + (kTile - 1) * (fmin(c, 0.0) + fmin(s, 0.0)) - 1e-3);
            const int row = (int) fmin(fmax(lo, (double) -kPad), (double) W) + kPad;
            par[chunk & 1][tid] = make_float4(sc.x, sc.y, (float) (u0 - lo), __int_as_float(row));
        }
    };
    const unsigned lds_base = (unsigned) (unsigned long) (LdsChar *) buf;
    // Pieces of 1 KB of a quad, [angle][group][plane][3]: piece k NW + wv is this wave's k-th.
    // Its source is scalar but for the lane's 16 bytes; the quad's rows wait in a register
    // (lane a: angle a's), so that no load waits for an LDS read.
    long piece[LOADS];
    int piece_angle[LOADS];
#pragma unroll
    for (int k = 0; k < LOADS; k++) {
        const int L = k * NW + wv;
        const int sub = L / 3, part = L - 3 * sub;
        const int a = sub / (NG * PL), gp = sub - a * (NG * PL);
        const int gi = gp / PL, pl = gp - gi * PL;
        piece[k] = (long) gi * group_bytes + ((long) (a * PL + pl) * Wp) * kRow + part * 1024;
        piece_angle[k] = a;
    }
    auto rows_of = [&](int q) {
        return __float_as_int(par[(q >> 4) & 1][(4 * q + (lane & 3)) & (kParChunk - 1)].w);
    };
    auto stage = [&](int q, int rows) {
        const char *src = base + (long) (p0 + 4 * q) * (PL * Wp) * kRow;
        const unsigned dst = lds_base + (q & 1) * QUAD + wv * 1024;
#pragma unroll
        for (int k = 0; k < LOADS; k++)
            load_lds(dst + k * NW * 1024, src + piece[k] + __builtin_amdgcn_readlane(rows, piece_angle[k]) * kRow,
                     lane * 16);
    };

    const int l16 = lane & 15, g = lane >> 4;
    const int wb = wv * BPW;  // this wave's first block; 8 blocks in a row of the tile
    const float xx = (float) (4 * (wb & 7) + (l16 & 3)), yy = (float) (l16 >> 2);
    // read address of this lane within a quad: angle g, entry l16 / 4, 4 slices of the first
    // (second at odd angles) half row; the rows of four entries and the halves of two angles then
    // cover all 64 banks
    const int rbase = g * (NG * PL * kPlane) + (l16 >> 2) * kRow + (l16 & 3) * 8 + (g & 1) * 32;
    // block (l16 mod BPW) of this wave, for the window starts
    const float cbx = (float) (4 * ((wb + (l16 & (BPW - 1))) & 7)), cby = (float) (4 * ((wb + (l16 & (BPW - 1))) >> 3));

    float4_t acc[BPW][NG * NT];
#pragma unroll
    for (int i = 0; i < BPW; i++)
#pragma unroll
        for (int n = 0; n < NG * NT; n++) acc[i][n] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};

    const int sel_base = (int) (unsigned) (unsigned long) (LdsChar *) seltab;
    // Geometry of this lane's angle in a quad of angles.
    struct Quad {
        float c, t[(BPW + 7) / 8];  // u of voxel x is c x + t[row]
        int sel0, j0r;              // of block l16: selector table less its window start, read address
    };
    auto par_of = [&](int q) { return par[(q >> 4) & 1][(4 * q + g) & (kParChunk - 1)]; };
    auto quad_of = [&](int q, const float4 &pr) {
        Quad r;
        const float s = pr.x, a = pr.z;
        r.c = pr.y;
        // the detector position of the block's corner, formed by the same operations as the
        // voxels' (so no voxel lies below it)
        const float um = fmaf(cbx + (r.c < 0.0f ? 3.0f : 0.0f), r.c, fmaf(cby + (s < 0.0f ? 3.0f : 0.0f), s, a));
        r.sel0 = sel_base - ((int) um << 4);
        r.j0r = (int) um * kRow + (int) lds_base + (q & 1) * QUAD;
#pragma unroll
        for (int k = 0; k < (BPW + 7) / 8; k++) r.t[k] = fmaf((float) (4 * ((wb >> 3) + k)) + yy, s, a);
        return r;
    };

    // One software pipeline over all steps (a block and a group of 32 slices) of all quads: the
    // selectors and weights of a block are formed two blocks ahead, the data of a step is read
    // one step ahead, across the barrier between two quads.
    uint4_t sel[2];
    unsigned ph[2], pl[2];
    half8_t d[2][NT][PL];
    auto weights = [&](auto bc, const Quad &qd) {
        constexpr int B = decltype(bc)::value;
        const float u = fmaf((float) (4 * (B & 7)) + xx, qd.c, qd.t[B >> 3]);
        const float f = __builtin_amdgcn_fractf(u);
        sel[B & 1] = *(const LdsUint4 *) (uintptr_t) (unsigned) (((int) u << 4) + row_bcast<B>(qd.sel0));
        // weights (1 - f, f) in f16, and what is left of them
        const float e = 1.0f - f;
        ph[B & 1] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_pkrtz(e, f));
        pl[B & 1] = residue(ph[B & 1], e, f);
    };
    unsigned o0 = 0, o1 = 0;  // first and second half row of the block being read
    auto load = [&](auto sc, const Quad &qd) {
        constexpr int ST = decltype(sc)::value, B = ST / NG, GI = ST % NG;
        if constexpr (GI == 0) {
            o0 = (unsigned) (rbase + row_bcast<B>(qd.j0r));
            o1 = o0 ^ 32;
        }
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
            for (int p = 0; p < PL; p++) {
                const LdsChar *r = (const LdsChar *) (uintptr_t) (n ? o1 : o0) + (GI * PL + p) * kPlane;
                const short4_t v0 = read_tr(r), v1 = read_tr(r + 4 * kRow);
                d[ST & 1][n][p] = __builtin_bit_cast(half8_t, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
            }
    };

    parameters(0);
    __syncthreads();
    stage(0, rows_of(0));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (nq > 1) stage(1, rows_of(1));
    Quad cur = quad_of(0, par_of(0));
    weights(std::integral_constant<int, 0>(), cur);
    weights(std::integral_constant<int, 1>(), cur);
    load(std::integral_constant<int, 0>(), cur);
    for (int q = 0; q < nq; q++) {
        if ((q & 15) == 0 && 4 * (q + 16) < np) parameters((q >> 4) + 1);
        const float4 prn = par_of(min(q + 1, nq - 1));
        const int rows = rows_of(min(q + 2, nq - 1));
        Quad next;
        uint4_t wh, wl;
        static_for<0, BPW * NG>([&](auto sc) {
            constexpr int ST = decltype(sc)::value, B = ST / NG, GI = ST % NG;
            constexpr bool LAST = ST + 1 == BPW * NG;
            if constexpr (GI == 0) {
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    wh[k] = __builtin_amdgcn_perm(0u, ph[B & 1], sel[B & 1][k]);
                    wl[k] = __builtin_amdgcn_perm(0u, pl[B & 1], sel[B & 1][k]);
                }
                if constexpr (B + 2 == BPW) next = quad_of(q + 1, prn);
                if constexpr (B + 2 < BPW) weights(std::integral_constant<int, B + 2>(), cur);
                else weights(std::integral_constant<int, B + 2 - BPW>(), next);
            }
            if constexpr (!LAST) {
                load(std::integral_constant<int, ST + 1>(), cur);
            } else {
                // this quad's data is all in registers and the next one's has landed
                asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                if (q + 2 < nq) stage(q + 2, rows);
                load(std::integral_constant<int, 0>(), next);
            }
            __builtin_amdgcn_sched_barrier(0);  // the reads above go out before these products
            const half8_t ah = __builtin_bit_cast(half8_t, wh), al = __builtin_bit_cast(half8_t, wl);
            if constexpr (PL == 2)
#pragma unroll
                for (int n = 0; n < NT; n++)
                    acc[B][GI * NT + n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, d[ST & 1][n][PL - 1],
                                                                                 acc[B][GI * NT + n], 0, 0, 0);
#pragma unroll
            for (int n = 0; n < NT; n++)
                acc[B][GI * NT + n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, d[ST & 1][n][0],
                                                                             acc[B][GI * NT + n], 0, 0, 0);
#pragma unroll
            for (int n = 0; n < NT; n++)
                acc[B][GI * NT + n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, d[ST & 1][n][0],
                                                                             acc[B][GI * NT + n], 0, 0, 0);
        });
        cur = next;
    }

    // D of a block: lane holds voxels (0 .. 3, g) of slice l16
    const float fp = (float) p_norm;
    out += (long) blockIdx.y * part_pitch;
    // 16-byte stores need 4-byte alignment only; written as four, a slice of odd width took 24 slices
    // of 400 x 701 in f16 storage from 277 to 382 us
    typedef float vec_t __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
    for (int n = 0; n < NG * NT; n++) {
        const int sl = slice0 + (n / NT) * kSub + (n % NT) * 16 + l16;
        const float inv = sl < n_slices ? ldexpf(1.0f, -scale_exponent<PL>(maxbits[sl])) : 0.0f;
#pragma unroll
        for (int i = 0; i < BPW; i++) {
            const int x = x0 + 4 * ((wb + i) & 7), y = y0 + 4 * ((wb + i) >> 3) + g;
            if (sl >= n_slices || y >= roi_h) continue;
            float4_t r;
#pragma unroll
            for (int k = 0; k < 4; k++) r[k] = (acc[i][n][k] * inv) * 3.14159274101257324219f / fp;
            float *o = out + (long) sl * out_pitch + (long) y * roi_w + x;
            if (x + 3 < roi_w) {
                *(vec_t *) o = r;
            } else {
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (x + k < roi_w) o[k] = r[k];
            }
        }
    }
}

// Sum of n_split partial volumes of n floats, in split order.
__global__ __launch_bounds__(256) void sum_parts_kernel(const float *__restrict__ part, int n_split, long n, long plane,
                                                        float *__restrict__ out, long out_pitch)
{
    for (long i = (long) blockIdx.x * 256 + threadIdx.x; i < n; i += (long) gridDim.x * 256) {
        float s = part[i];
        for (int j = 1; j < n_split; j++) s += part[j * n + i];
        const long sl = i / plane;
        out[sl * out_pitch + (i - sl * plane)] = s;
    }
}

// Stored bytes of one 32-slice group.
size_t group_bytes(int W, int P, int planes)
{
    return (size_t) ((P + 3) / 4 * 4) * planes * (W + 2 * kPad) * kRow;
}

// How n slices go over the kernels: n64 units of 64 slices, then n32 of 32, then n16 of 16.
// Measured at 2048^2 pixels, 720 angles (TGUPS of full units): 64 slices 25.5, 32 slices 22.9,
// 16 slices 18.2 in f32 storage (16-bit: 37.8, 31.3, 22.4); the interpolating kernel's 8-slice
// tiles reach 11.9 (f16 16.7), so up to 8 leftover slices stay with it.
struct Units {
    int n64, n32, n16, slices;
};
Units units_of(int n)
{
    Units u = {n / 64, 0, 0, 0};
    int r = n % 64;
    if (r > 48) {
        u.n64++;
        r = 0;
    } else if (r > 16) {
        u.n32 = 1;
        r = r > 32 ? r - 32 : 0;
    }
    if (r > 8) {
        u.n16 = 1;
        r = 0;
    }
    u.slices = n - r;
    return u;
}

// Whether the units are faster than the interpolating kernel for them.  The layout reads and writes
// whole rows whatever the region of interest needs of them, so a small region of a wide detector
// does not pay for it; and up to 8 leftover slices take a launch of their own, too few workgroups
// to hide its 60 us.  Rates of updates (per us, in 1e6) as above, of the interpolating kernel as
// it reaches them on regions of 256 to 1024 pixels, and microseconds per 1e6 samples of the layout
// (a slice read, a slice of a group of 32 written).  Measured over 12 to 128 slices of 90 to 3000
// angles x 256 to 4096 pixels, whole and regions of 128 to 1024: 5 of 893 stacks go the slower way
// by more than 4%, at most 10%.
// In us, matrix cores / interpolating kernel, 64 slices of 1800 x 2048 in f32: 724 / 240 for 128^2
// pixels, 922 / 779 for 256^2, 1454 / 1748 for 384^2; 16 slices 479 / 451 for 384^2, 644 / 776 for 512^2;
// 100 slices (4 leftover) of 180 x 256 192 / 158.
bool pays(const ufomi_bp_stack &st, const Units &u)
{
    const bool f32 = st.dtype == UFOMI_F32;
    const double interp = st.dtype == UFOMI_F16 ? 14.5 : 10.8;
    const double r64 = f32 ? 25.5 : 37.8, r32 = f32 ? 22.9 : 31.3, r16 = f32 ? 18.2 : 22.4;
    const double read = f32 ? 1.77 : 1.0, write = f32 ? 0.64 : 1.1;
    const double updates = 1e-6 * ((st.roi_w + kTile - 1) / kTile) * ((st.roi_h + kTile - 1) / kTile) * kTile * kTile * st.P;
    const double layout = 1e-6 * st.P * st.W * (read * u.slices + write * ((u.slices + kSub - 1) / kSub * kSub));
    const double rest = u.slices < st.n_slices ? 60.0 + 0.6 * updates * 8 / interp : 0.0;
    return updates * (u.n64 * 64 / r64 + u.n32 * 32 / r32 + u.n16 * 16 / r16) + layout + rest <
           updates * ((st.n_slices + 7) / 8 * 8) / interp;
}

template <typename T, int PL> int run(ufomi_ctx *ctx, const T *sino, const ufomi_bp_stack &st, int *done)
{
    const Units all = units_of(st.n_slices);
    if (!all.slices || !pays(st, all)) return UFOMI_OK;
    const int n_slices = all.slices;
    const size_t gb = group_bytes(st.W, st.P, PL);
    const int groups_all = (n_slices + kSub - 1) / kSub;
    // whole units of 64 slices per chunk, unless one does not fit
    int per_chunk = (int) std::max<size_t>(1, std::min<size_t>({kWorkspace / gb, (size_t) groups_all, kGridY / kSub}));
    if (per_chunk > 1 && per_chunk < groups_all) per_chunk &= ~1;
    const int tiles_x = (st.roi_w + kTile - 1) / kTile, tiles_y = (st.roi_h + kTile - 1) / kTile;
    const long tiles = (long) tiles_x * tiles_y, plane = (long) st.roi_w * st.roi_h;
    // Few workgroups: split the angles (at least 64 each) towards two rounds of 512 workgroups,
    // into partial volumes summed in a fixed order.
    const Units first = units_of(std::min(per_chunk * kSub, n_slices));
    const long wgs = tiles * (2 * first.n64 + first.n32 + first.n16);
    int n_split = (int) std::max<long>(1, std::min<long>((1024 + wgs - 1) / wgs, std::min(8, st.P / 64)));
    const int P4 = (st.P + 3) / 4 * 4;
    const int p_chunk = n_split > 1 ? (P4 / 4 + n_split - 1) / n_split * 4 : P4;
    n_split = (P4 + p_chunk - 1) / p_chunk;
    // per slice: largest |v|, number of non-zero and of small samples
    const int words = per_chunk * kSub;
    const size_t head = (3 * (size_t) words * sizeof(unsigned) + 255) & ~(size_t) 255;
    const size_t rows_bytes = gb * per_chunk;
    const size_t part_bytes =
        n_split > 1 ? (size_t) n_split * std::min(per_chunk * kSub, n_slices) * plane * sizeof(float) : 0;
    char *ws = nullptr;
    int rc = ufomi_workspace(ctx, head + rows_bytes + part_bytes, (void **) &ws);
    if (rc == UFOMI_ERR_MEMORY) return UFOMI_OK;  // *done = 0: the caller has a path without it
    if (rc) return rc;
    unsigned *maxbits = (unsigned *) ws, *nonzero = maxbits + words, *small = nonzero + words;
    char *rows = ws + head;
    float *part = n_split > 1 ? (float *) (rows + rows_bytes) : nullptr;
    const int Wp = st.W + 2 * kPad;
    const long elems = (long) st.P * st.W;
    auto chunk = [&](int g0) {
        const int s0 = g0 * kSub, ns = std::min(per_chunk * kSub, n_slices - s0);
        const int ng = (ns + kSub - 1) / kSub;
        const T *in = sino + (size_t) s0 * st.sino_pitch;
        float *out = st.out + (size_t) s0 * st.out_pitch;
        hipLaunchKernelGGL(clear_kernel, dim3((3 * words + 255) / 256), dim3(256), 0, ctx->stream, maxbits,
                           3 * words);
        UFOMI_CHECK_LAUNCH();
        const unsigned mb = (unsigned) std::min<long>((elems + 8191) / 8192, 64);
        hipLaunchKernelGGL(absmax_kernel<T>, dim3(mb, ns), dim3(256), 0, ctx->stream, in, (long) st.sino_pitch, elems,
                           maxbits, nonzero);
        UFOMI_CHECK_LAUNCH();
        hipLaunchKernelGGL((split_kernel<T, PL>), dim3((Wp + 63) / 64, P4, ng), dim3(256), 0, ctx->stream, in,
                           (long) st.sino_pitch, st.W, st.P, Wp, ns, maxbits, nonzero, small, (uint4_t *) rows,
                           (long) (gb / 16));
        UFOMI_CHECK_LAUNCH();
        // `count` slices from slice `first` of the chunk, `unit` per workgroup
        auto launch = [&](auto kernel, int threads, int unit, int first, int count) {
            if (count <= 0) return (int) UFOMI_OK;
            const long blocks = tiles * ((count + unit - 1) / unit);
            hipLaunchKernelGGL(kernel, dim3((unsigned) blocks, (unsigned) n_split), dim3(threads), 0, ctx->stream,
                               rows + (size_t) (first / kSub) * gb, (long) gb, Wp, st.W, st.P, st.trig, st.axis,
                               st.roi_x, st.roi_y, st.roi_w, st.roi_h, count, maxbits + first,
                               part ? part + (size_t) first * plane : out + (size_t) first * st.out_pitch,
                               part ? plane : (long) st.out_pitch, part ? (long) ns * plane : 0L, tiles_x, tiles_y,
                               p_chunk, st.P);
            UFOMI_CHECK_LAUNCH();
            return (int) UFOMI_OK;
        };
        const Units u = units_of(ns);
        const int a = std::min(64 * u.n64, ns), b = std::min(a + 32 * u.n32, ns), e = std::min(b + 16 * u.n16, ns);
        if (int rc = launch(bp_mfma_kernel<2, 2, PL, 8>, 512, 64, 0, a)) return rc;
        if (int rc = launch(bp_mfma_kernel<1, 2, PL, 4>, 256, 32, a, b - a)) return rc;
        if (int rc = launch(bp_mfma_kernel<1, 1, PL, 4>, 256, 16, b, e - b)) return rc;
        if (part) {
            const long total = plane * ns;
            hipLaunchKernelGGL(sum_parts_kernel, dim3((unsigned) std::min<long>((total + 255) / 256, 8192)), dim3(256),
                               0, ctx->stream, part, n_split, total, plane, out, (long) st.out_pitch);
            UFOMI_CHECK_LAUNCH();
        }
        return ufomi_bp_left_out(ctx, st, s0, ns, a, b, maxbits);
    };
    for (int g0 = 0; g0 < groups_all && !rc; g0 += per_chunk) rc = chunk(g0);
    // also where a launch failed: those before it use the workspace
    const int end = ufomi_workspace_done(ctx);
    if (!rc) rc = end;
    if (!rc) *done = n_slices;
    return rc;
}

}  // namespace

int ufomi_bp_mfma(ufomi_ctx *ctx, const ufomi_bp_stack &st, int *done)
{
    *done = 0;
    // no workspace can be had under capture, and none shared with a captured graph is safe
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    UFOMI_HIP(hipStreamIsCapturing(ctx->stream, &cap));
    if (cap != hipStreamCaptureStatusNone) return UFOMI_OK;
    if (group_bytes(st.W, st.P, st.dtype == UFOMI_F32 ? 2 : 1) > kGroupMax || st.P > kGridY / 4 * 4) return UFOMI_OK;
    const long tiles = (long) ((st.roi_w + kTile - 1) / kTile) * ((st.roi_h + kTile - 1) / kTile);
    if (tiles * ((st.n_slices + 15) / 16) > 0x7fffffffL) return UFOMI_OK;
    switch (st.dtype) {
    case UFOMI_F16: return run<__half, 1>(ctx, (const __half *) st.sino, st, done);
    case UFOMI_BF16: return run<__hip_bfloat16, 1>(ctx, (const __hip_bfloat16 *) st.sino, st, done);
    default: return run<float, 2>(ctx, (const float *) st.sino, st, done);
    }
}
