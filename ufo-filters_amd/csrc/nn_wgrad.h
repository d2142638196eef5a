// Weight gradients of the 3x3 convolutions on NHWC activations as they are (unet.hip): no
// channel-major copies, every staged row is used for all nine taps.
//
// dW[co][ky][kx][ci] = sum over pixels of g[y][x][co] in[y + ky - 1][x + kx - 1][ci] is a product
// whose K runs over pixels, while NHWC has the channels next to each other.  ds_read_b64_tr_b16
// transposes on the way from LDS: 16 lanes address 4 pixels x 16 channels and receive 4 pixels of
// one channel each, which is a fragment of v_mfma_f32_16x16x32_bf16.  A tap's column shift is
// then an LDS offset and its row shift a choice of rows, so an input row is read from memory and
// its three fragments sets from LDS once, against the three gradient rows kept in registers.
//
// A wave owns 32 x 32 channels of all nine taps (144 accumulators) and walks down R rows of a
// strip of 32 pixels; the 8 waves of a workgroup take different strips and row chunks, and their
// sums meet in LDS, so only one partial per workgroup goes to memory.  Waves share nothing before
// that: each has its own ring of 4 rows in LDS, filled by global_load_lds three rows ahead.
// Bias gradients are one more product with ones, in the tiles of the first input channels.
//
// Bound by the matrix cores' issue (36 products of 16 cycles a row and wave) and, for 32
// channels, by reading g and in (128 B per pixel).  8 images of 256^2 with 64 x 64 channels at
// half size (9.7 GFLOP): 20.5 us, against 58 us for the split-K product on channel-major copies,
// 31 us for making the copies, 18 us for the bias sums and 17 us for adding the partials; the
// partials now add in 5 us (1 per workgroup instead of 512 in all).
#pragma once

#include "nn_gemm.h"

namespace nn {

constexpr int kWgWaves = 8, kWgRing = 4;
constexpr int kWgG = 32 * 64, kWgX = 34 * 64, kWgSlot = kWgG + kWgX;  // bytes of a row of each operand

__device__ const f32x4 wg_zeros = {0.0f, 0.0f, 0.0f, 0.0f};

struct Wgrad3 {
    View<const bf16> g, in;
    int lh, lw;     // image of 2^lh x 2^lw pixels, lw >= 5
    int lr;         // 2^lr rows per unit, lr <= lh
    int cin, cout;  // multiples of 32
    int units;      // strips of 32 pixels x 2^lr rows
    int splits;     // workgroups per tile of channels; a wave takes every (8 splits)-th unit
    float *part;    // [splits][cout][9][cin], then cout bias sums, per split
};

typedef __attribute__((address_space(3))) char wg_lds_char;

// The fragment of 32 pixels x 16 channels at LDS address a: pixels 4 q .. 4 q + 3 and 16 + the same.
__device__ __forceinline__ bf16x8 wg_fragment(wg_lds_char *a)
{
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    typedef __attribute__((address_space(3))) s16x4 LdsTile;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsTile *) a);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsTile *) (a + 1024));
    return __builtin_bit_cast(bf16x8, (s16x8) __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

__global__ __launch_bounds__(kWgWaves * 64) void wgrad3_kernel(Wgrad3 op)
{
    __shared__ __align__(16) char wg_lds[kWgWaves * kWgRing * kWgSlot];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, q = lane >> 4;
    const int split = blockIdx.x % op.splits, tile = blockIdx.x / op.splits;
    const int tiles_m = op.cout / 32, co0 = (tile % tiles_m) * 32, ci0 = (tile / tiles_m) * 32;
    const int R = 1 << op.lr, H = 1 << op.lh, W = 1 << op.lw;
    const bool bias = ci0 == 0;

    f32x4 acc[3][3][2][2], accb[2];
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
        for (int k = 0; k < 4; k++) acc[t / 3][t % 3][k >> 1][k & 1] = zero;
    accb[0] = accb[1] = zero;

    for (int unit = split * kWgWaves + wave; unit < op.units; unit += op.splits * kWgWaves) {
        const int sl = op.lw - 5, cl = op.lh - op.lr;
        const int x0 = (unit & ((1 << sl) - 1)) * 32, ya = ((unit >> sl) & ((1 << cl) - 1)) << op.lr;
        const long img = unit >> (sl + cl);
        wg_lds_char *ring = (wg_lds_char *) wg_lds + wave * (kWgRing * kWgSlot);
        // Slot of 16 bytes e of a staged row: pixel e / 4, channels 8 (e % 4 ^ 2 (pixel / 4 % 2)):
        // any 8 consecutive pixels then have their 16 channels of a fragment in different banks.
        const int px = lane >> 2, ch = 8 * ((lane & 3) ^ ((px >> 2 & 1) << 1));
        const bf16 *gp = op.g.at((((img << op.lh) + ya) << op.lw) + x0 + px, co0 + ch);
        const bf16 *xp = op.in.at((((img << op.lh) + ya - 1) << op.lw) + x0 - 1 + px, ci0 + ch);
        const long g_row = (long) op.g.cs << op.lw, x_row = (long) op.in.cs << op.lw;
        const bool left = x0 > 0 || px > 0, right = x0 + 32 < W || px == 0;
        // Rows of step i: gradient row ya + i and input row ya - 1 + i; what is outside reads zeros.
        auto stage = [&](int i) {
            const unsigned dst = (unsigned) (uintptr_t) (ring + (i % kWgRing) * kWgSlot);
            const bool gok = i < R, xok = i < R + 2 && ya - 1 + i >= 0 && ya - 1 + i < H;
            const bf16 *gs = gp + i * g_row, *xs = xp + i * x_row;
            const void *z = &wg_zeros;
            load_lds_async(dst, gok ? gs : z);
            load_lds_async(dst + 1024, gok ? gs + 16 * op.g.cs : z);
            load_lds_async(dst + kWgG, xok && left ? xs : z);
            load_lds_async(dst + kWgG + 1024, xok ? xs + 16 * op.in.cs : z);
            // pixels 32 and 33 (one lane in four of 8: the same channels as pixels 0 and 1)
            if (lane < 8) load_lds_async(dst + kWgG + 2048, xok && right ? xs + 32 * op.in.cs : z);
        };
        // Fragment addresses within a slot: this lane's pixel 4 q + l16 / 4, 4 channels.
        auto address = [&](int p) { return p * 64 + 16 * ((l16 & 3) >> 1) + 8 * (l16 & 1) + 32 * (p >> 2 & 1); };
        const unsigned ga = address(4 * q + (l16 >> 2));
        unsigned xa[3];
#pragma unroll
        for (int kx = 0; kx < 3; kx++) xa[kx] = kWgG + address(4 * q + (l16 >> 2) + kx);
        bf16x8 ones;
#pragma unroll
        for (int e = 0; e < 8; e++) ones[e] = (bf16) 1.0f;

        bf16x8 g0[2], g1[2], g2[2];  // gradient rows ya + i, ya + i - 1, ya + i - 2
        g0[0] = g0[1] = g1[0] = g1[1] = g2[0] = g2[1] = zero8();
        stage(0);
        stage(1);
        stage(2);
        for (int i = 0; i < R + 2; i++) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // row i - 1's slot has been read
            stage(i + 3);
            asm volatile("s_waitcnt vmcnt(15)" ::: "memory");  // 3 rows of 5 loads later than row i
            wg_lds_char *slot = ring + (i % kWgRing) * kWgSlot;
            const bool in0 = i < R, in1 = i >= 1 && i < R + 1, in2 = i >= 2;
            const bool xin = ya - 1 + i >= 0 && ya - 1 + i < H;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                g2[h] = g1[h];
                g1[h] = g0[h];
            }
            bf16x8 x[3][2];
#pragma unroll
            for (int kx = 0; kx < 3; kx++)
#pragma unroll
                for (int h = 0; h < 2; h++) x[kx][h] = wg_fragment(slot + (xa[kx] ^ (32 * h)));
#pragma unroll
            for (int h = 0; h < 2; h++) g0[h] = wg_fragment(slot + (ga ^ (32 * h)));
            auto products = [&](f32x4(&a)[3][2][2], const bf16x8(&gr)[2]) {
#pragma unroll
                for (int kx = 0; kx < 3; kx++)
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        a[kx][k >> 1][k & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gr[k >> 1], x[kx][k & 1],
                                                                                       a[kx][k >> 1][k & 1], 0, 0, 0);
            };
            // input row r meets gradient row r + 1 at ky = 0, r at ky = 1, r - 1 at ky = 2
            if (in2 && xin) products(acc[2], g2);
            if (in1 && xin) products(acc[1], g1);
            if (in0 && xin) products(acc[0], g0);
            if (in0 && bias)
#pragma unroll
                for (int h = 0; h < 2; h++)
                    accb[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(g0[h], ones, accb[h], 0, 0, 0);
        }
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // the ring is used again below
    }

    // Sums of the 8 waves: at step t wave w adds tap (w + t) % 9 to the workgroup's sums, so every
    // tap is added in a fixed order and by one wave at a time.
    f32x4 *sum = reinterpret_cast<f32x4 *>(wg_lds);  // [tap][tile][lane]
    float *bsum = reinterpret_cast<float *>(sum + 9 * 4 * 64);  // [wave][32]
    __syncthreads();
    for (int t = 0; t < 9; t++) {
        const int own = (wave + t) % 9;
        const bool first = t == 0 || (t == 1 && own == 8);
#pragma unroll
        for (int p = 0; p < 9; p++)
            if (p == own)
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    f32x4 v = acc[p / 3][p % 3][k >> 1][k & 1];
                    if (!first) v += sum[(p * 4 + k) * 64 + lane];
                    sum[(p * 4 + k) * 64 + lane] = v;
                }
        __syncthreads();
    }
    if (bias && l16 == 0)
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int e = 0; e < 4; e++) bsum[wave * 32 + 16 * h + 4 * q + e] = accb[h][e];
    __syncthreads();
    const long len = 9L * op.cin * op.cout + op.cout;
    float *dst = op.part + split * len;
    for (int e = threadIdx.x; e < 9 * 4 * 64; e += kWgWaves * 64) {
        const int tap = e >> 8, k = e >> 6 & 3, ln = e & 63;
        const f32x4 v = sum[e];
#pragma unroll
        for (int c = 0; c < 4; c++)
            dst[((co0 + 16 * (k >> 1) + 4 * (ln >> 4) + c) * 9L + tap) * op.cin + ci0 + 16 * (k & 1) + (ln & 15)] = v[c];
    }
    if (bias && threadIdx.x < 32) {
        float s = 0.0f;
        for (int w = 0; w < kWgWaves; w++) s += bsum[w * 32 + threadIdx.x];
        dst[9L * op.cin * op.cout + co0 + threadIdx.x] = s;
    }
}

// The first convolution (one input channel, 32 outputs): the 9 taps are the columns of one
// product, column 9 holds ones and gives the bias sums.  A wave takes R rows of a 32-pixel strip;
// g goes through LDS for the transposing read, the taps' pixels come straight from the image
// (L1), both a row ahead.  Bound by reading g (64 B per pixel): 12 us for 8 images of 256^2, against
// 60 us with the generic product and 18 us for the bias.
struct WgradFirst {
    View<const bf16> g;
    const bf16 *img;  // [pixels]
    int lh, lw, lr, units, splits;
    float *part;      // [splits][32 x 9 weights, 32 biases]
};

__global__ __launch_bounds__(kWgWaves * 64) void wgrad_first_kernel(WgradFirst op)
{
    __shared__ __align__(16) char rows[kWgWaves][2][kWgG];
    __shared__ f32x4 sums[kWgWaves][2][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, q = lane >> 4;
    const int R = 1 << op.lr, H = 1 << op.lh, W = 1 << op.lw;
    f32x4 acc[2];
    acc[0] = acc[1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int unit = blockIdx.x * kWgWaves + wave; unit < op.units; unit += op.splits * kWgWaves) {
        const int sl = op.lw - 5, cl = op.lh - op.lr;
        const int x0 = (unit & ((1 << sl) - 1)) * 32, ya = ((unit >> sl) & ((1 << cl) - 1)) << op.lr;
        const long img = unit >> (sl + cl);
        const int px = lane >> 2, ch = 8 * ((lane & 3) ^ ((px >> 2 & 1) << 1));
        const bf16 *gp = op.g.at((((img << op.lh) + ya) << op.lw) + x0 + px, ch);
        const bf16 *image = op.img + (img << (op.lh + op.lw));
        const int ky = l16 / 3, kx = l16 % 3;
        bf16x8 ga, gb, b;
        auto fetch = [&](int y) {
            const bf16 *gs = gp + (((long) (y - ya) * op.g.cs) << op.lw);
            ga = ld8(gs);
            gb = ld8(gs + 16 * op.g.cs);
            const int yy = y + ky - 1;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int xx = x0 + kx - 1 + 4 * q + (e & 3) + 16 * (e >> 2);
                const bool ok = l16 < 9 && yy >= 0 && yy < H && xx >= 0 && xx < W;
                const bf16 v = image[ok ? ((long) yy << op.lw) + xx : 0];
                b[e] = l16 == 9 ? (bf16) 1.0f : ok ? v : (bf16) 0.0f;
            }
        };
        const int p = 4 * q + (l16 >> 2);
        const int a = p * 64 + 16 * ((l16 & 3) >> 1) + 8 * (l16 & 1) + 32 * (p >> 2 & 1);
        fetch(ya);
        for (int i = 0; i < R; i++) {
            char *row = rows[wave][i & 1];
            *reinterpret_cast<bf16x8 *>(row + lane * 16) = ga;
            *reinterpret_cast<bf16x8 *>(row + 1024 + lane * 16) = gb;
            const bf16x8 taps = b;
            if (i + 1 < R) fetch(ya + i + 1);
            // a wave's LDS accesses are in order: the write above is seen by the reads below
            asm volatile("" ::: "memory");
            wg_lds_char *base = (wg_lds_char *) row;
#pragma unroll
            for (int h = 0; h < 2; h++)
                acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wg_fragment(base + (a ^ (32 * h))), taps, acc[h], 0, 0,
                                                                 0);
        }
    }
    sums[wave][0][lane] = acc[0];
    sums[wave][1][lane] = acc[1];
    __syncthreads();
    if (threadIdx.x >= 128) return;
    const int h = threadIdx.x >> 6;
    f32x4 s = sums[0][h][lane];
    for (int w = 1; w < kWgWaves; w++) s += sums[w][h][lane];
    float *dst = op.part + blockIdx.x * 320L;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int co = 16 * h + 4 * q + e;
        if (l16 < 9) dst[co * 9 + l16] = s[e];
        if (l16 == 9) dst[288 + co] = s[e];
    }
}

}  // namespace nn
