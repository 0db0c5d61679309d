// conv_fp32.hip — the FP32 "plain" form of Leela's policy and value nets.
//
// FP32 convolution on the 16-bit matrix cores (conv_split). Every FP32 value
// is written as the sum of three BF16 values (round to nearest each time:
// 8 + 8 + 8 bits and their signs hold the 24 bits exactly from 2^-103 up;
// below that the smallest part can be a BF16 subnormal, which the matrix unit
// takes as 0), and a product is
// the sum of the six largest partial products, each exact in FP32; the two
// of up to 2^-25 of it each that are left out make 2^-24 at most (random
// pairs: 2^-24.04, past 2^-25 for one in a thousand):
//   a b = a1 b1 + a1 b2 + a2 b1 + a2 b2 + a1 b3 + a3 b1 + O(2^-24 a b).
// Sums are FP32 throughout (v_mfma_f32_16x16x32_bf16 adds 32 products with
// fewer roundings than an FP32 chain has), activations stay FP32 in memory.
// Against 64 bits the nets' outputs are no further off than with FP32 MFMA
// (policy probabilities of 96 boards 3.7e-6 against 5.1e-6, a trained net's
// logits 3.7e-6 against 4.2e-6). The FP32 matrix unit runs at 1/16 of the
// BF16 rate, so six products are 2.7 times its peak: 1024 boards through
// the policy net take 5.12 ms (240 TFLOP/s of FP32 products), against 15.9
// on FP32 MFMA (77 TFLOP/s of 157).
//
// The product is the one that the reference forms with im2col + sgemm
// (Network.cpp:344-393, Im2Col.h:9-50). Bias, the activation (ELU,
// Network.cpp:382-392; or ReLU / none for Caffe nets) and an optional batch
// normalisation of the activated output (Network.cpp:427-448) are fused
// into the epilogue. Activations between convs: [n][361][C], C rounded up to
// 32 channels (the extra ones zero).
#include <type_traits>

#include "lz_conv_tile.h"
#include "lz_internal.h"

namespace lz {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kThreads = 256;           // 4 waves
constexpr int kS = 19, kP = kS * kS;    // the nets' board

__device__ __forceinline__ float elu(float v) {
    return v > 0.0f ? v : (expf(v) - 1.0f);
}

__device__ __forceinline__ float activate(float v, int act) {
    if (act == kActElu) return elu(v);
    if (act == kActRelu) return v > 0.0f ? v : 0.0f;
    return v;
}

// The three BF16 parts of eight FP32 values. (Values past BF16's largest,
// 3.39e38, take that as their first part. The third part of an infinity is
// NaN, and so is every sum that it is in: see conv_split.)
__device__ __forceinline__ void split3(const float (&x)[8], bf16x8 (&p)[3]) {
    constexpr float kMax = 3.3895313892515355e38f;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const __bf16 h = (__bf16)__builtin_amdgcn_fmed3f(x[e], -kMax, kMax);
        const float r = x[e] - (float)h;
        const __bf16 m = (__bf16)r;
        p[0][e] = h;
        p[1][e] = m;
        p[2][e] = (__bf16)(r - (float)m);
    }
}

// Sums of products with scaled weights: which cannot stand (see conv_split).
struct SumProbe {
    uint32_t small = 0xffffffffu;  // least twice the bits of a sum, less 1
    float bad = 0.f;               // NaN if a sum is not finite
    __device__ __forceinline__ void scaled(float v) {
        const uint32_t b = (__float_as_uint(v) << 1) - 1;
        small = b < small ? b : small;
    }
    __device__ __forceinline__ void sum(float v) { bad = fmaf(v, 0.f, bad); }
    __device__ __forceinline__ bool again() const {
        return bad != bad || small < (47u << 24) - 1;  // 0 < |v| < 2^-80
    }
};

// One conv. A workgroup computes a band of R image rows of one board (10
// rows, NTW = 6, or 5, NTW = 3) for 2 * MTW m-tiles of 16 output channels:
// its four waves are 2 (channels) x 2 (pixels), each MTW m-tiles x NTW
// column tiles of 16 pixels. Per chunk of 32 input channels the band's rows
// and halo are split and staged in LDS, HWC, the parts of a pixel side by
// side (NB = 3 parts of 32 channels; byte planes are exact in one, NB = 1),
// then F * F k-steps follow. Weights: [chunk][tap][part][m-tile][lane][8].
//
// Weights are over their output channel's scale. A wave with a sum that is
// not finite, or below 2^-80 and not 0, forms its sums again in FP32 (the
// matrix unit's 16x16x4, the plain weights). The partial products of an
// infinity, or of a product past FP32's range, have both signs and add up to
// NaN where FP32 has an infinity. And what inputs below 2^-103 lack, 2^-126
// each, is 2^-111 at most over a sum's terms, less than 2^-24 of any sum from
// 2^-80 up. (Weights below 2^-103 of their channel's largest lack bits for
// good; that shows only where inputs make up for 30 orders of magnitude.)
// Ordinary nets never get there.
//
// Bound: the matrix cores, six products a term. The order of the products
// gives every operand's reload a group of MFMAs or more before its next
// use. Small pieces (few MFMAs a step) keep F steps of weights on the way
// and load the next chunk's values under this one's MFMAs (policy net, one
// board: 310 us without, 216 with).
template <int F, int NB, int MTW, int NTW>
__global__ __launch_bounds__(kThreads, MTW * NTW > 3 ? 2 : 3) void conv_split(
    const void *__restrict__ in, const bf16x8 *__restrict__ wpk,
    const float *__restrict__ wscale, const float *__restrict__ wplain,
    const float *__restrict__ bias, float *__restrict__ out, int cin,
    int chunks, int cout, int cstride, int mtiles, ConvEpilogue epi) {
    constexpr int R = NTW == 6 ? 10 : 5, BANDS = (kS + R - 1) / R;
    constexpr int W = kS + F - 1, PS = NB * 32 + 16;
    constexpr int RP = W * PS + row_pad(PS, F - 1);
    constexpr int FF = F * F;
    constexpr bool kSmall = NTW == 3 && MTW <= 2;
    // k-steps of weights held (a divisor of F * F, as registers allow).
    constexpr int D = kSmall && (F == 3 || MTW == 1) ? F : 1;
    constexpr int TASKS = ((R + F - 1) * W * 4 + kThreads - 1) / kThreads;
    static_assert(R * kS <= 2 * NTW * 16, "column tiles cover the band");
    __shared__ __attribute__((aligned(16))) __bf16 tile[(R + F - 1) * RP];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int board = blockIdx.x / BANDS, y0 = blockIdx.x % BANDS * R;
    const int rows = y0 + R < kS ? R : kS - y0, npx = rows * kS;
    const int mt0 = (blockIdx.y * 2 + (w & 1)) * MTW;
    const int g8 = (lane >> 4) * 8;

    int pb[NTW], pix[NTW];
#pragma unroll
    for (int t = 0; t < NTW; t++) {
        const int j = ((w >> 1) * NTW + t) * 16 + (lane & 15);
        pix[t] = j < npx ? y0 * kS + j : -1;
        // A lane past the band reads a pixel a multiple of 16 before it.
        const int jj = j < npx ? j : j - ((j - npx) / 16 + 1) * 16;
        pb[t] = (jj / kS) * RP + (jj % kS) * PS + g8;
    }
    f32x4 acc[MTW][NTW];
#pragma unroll
    for (int m = 0; m < MTW; m++)
#pragma unroll
        for (int t = 0; t < NTW; t++) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};

    // Weights of k-step s (over chunks and taps), part p, into set d. Tiles
    // past the last m-tile re-read it and are not stored.
    const int steps = chunks * FF;
    int mt[MTW];
#pragma unroll
    for (int m = 0; m < MTW; m++)
        mt[m] = (mt0 + m < mtiles ? mt0 + m : mtiles - 1) * 64 + lane;
    bf16x8 a[D][3][MTW], b[NB][NTW];
    auto load_a = [&](int d, int s, int p) {
        s = s < steps ? s : steps - 1;
        const bf16x8 *at = wpk + (size_t)(s * 3 + p) * mtiles * 64;
#pragma unroll
        for (int m = 0; m < MTW; m++) a[d][p][m] = at[mt[m]];
    };
    auto load_b = [&](int tap, int p) {
        tap = tap < FF ? tap : FF - 1;
        const __bf16 *at = tile + (tap / F) * RP + (tap % F) * PS + p * 32;
#pragma unroll
        for (int t = 0; t < NTW; t++)
            b[p][t] = *(const bf16x8 *)(at + pb[t]);
    };
    auto mul = [&](int d, int pa, int pbk) {
#pragma unroll
        for (int m = 0; m < MTW; m++)
#pragma unroll
            for (int t = 0; t < NTW; t++)
                acc[m][t] =
                    Op<__bf16>::mfma(a[d][pa][m], b[pbk][t], acc[m][t]);
    };
    // Task k of a chunk's staging: eight channels of a point of the band's
    // frame (zeros off the board), as values (float input) or one part.
    auto fetch = [&](int chunk, int k, float (&v)[8]) {
        const int i = tid + k * kThreads;
        const int c8 = (i & 3) * 8, q = i >> 2;
        const int y = y0 - F / 2 + q / W, x = q % W - F / 2;
        const bool on = q < (R + F - 1) * W && y >= 0 && y < kS && x >= 0 &&
                        x < kS;
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = 0.f;
        if (!on) return;
        if (NB == 1) {
            const int c = chunk * 32 + c8;
            const uint8_t *src =
                (const uint8_t *)in + ((size_t)board * cin + c) * kP + y * kS + x;
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (c + e < cin) v[e] = (float)src[e * kP];
        } else {
            const f32x4 *src =
                (const f32x4 *)((const float *)in +
                                ((size_t)board * kP + y * kS + x) *
                                    (chunks * 32) +
                                chunk * 32 + c8);
            const f32x4 lo = src[0], hi = src[1];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v[e] = lo[e];
                v[4 + e] = hi[e];
            }
        }
    };
    auto put = [&](int k, const float (&v)[8]) {
        const int i = tid + k * kThreads, q = i >> 2;
        if (q >= (R + F - 1) * W) return;
        __bf16 *dst = tile + (q / W) * RP + (q % W) * PS + (i & 3) * 8;
        bf16x8 parts[3];
        split3(v, parts);
#pragma unroll
        for (int p = 0; p < NB; p++) *(bf16x8 *)(dst + p * 32) = parts[p];
    };
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
        for (int p = 0; p < 3; p++) load_a(d, d, p);

    float next[kSmall ? TASKS : 1][8];
    if constexpr (kSmall) {
#pragma unroll
        for (int k = 0; k < TASKS; k++) fetch(0, k, next[k]);
    }
    for (int chunk = 0; chunk < chunks; chunk++) {
        __syncthreads();
        if constexpr (kSmall) {
#pragma unroll
            for (int k = 0; k < TASKS; k++) put(k, next[k]);
            if (chunk + 1 < chunks) {
#pragma unroll
                for (int k = 0; k < TASKS; k++) fetch(chunk + 1, k, next[k]);
            }
        } else {
            for (int k = 0; k < TASKS; k++) {
                fetch(chunk, k, next[0]);
                put(k, next[0]);
            }
        }
        __syncthreads();
#pragma unroll
        for (int p = 0; p < NB; p++) load_b(0, p);
        for (int tap0 = 0; tap0 < FF; tap0 += D) {
#pragma unroll
            for (int d = 0; d < D; d++) {
                const int tap = tap0 + d, s = chunk * FF + tap + D;
                if constexpr (NB == 3) {
                    mul(d, 0, 2);
                    load_b(tap + 1, 2);
                    mul(d, 0, 1);
                    mul(d, 0, 0);
                    load_a(d, s, 0);
                    mul(d, 1, 0);
                    mul(d, 1, 1);
                    load_a(d, s, 1);
                    load_b(tap + 1, 1);
                    mul(d, 2, 0);
                    load_a(d, s, 2);
                    load_b(tap + 1, 0);
                } else {
                    mul(d, 0, 0);
                    load_a(d, s, 0);
                    mul(d, 1, 0);
                    load_a(d, s, 1);
                    mul(d, 2, 0);
                    load_a(d, s, 2);
                    load_b(tap + 1, 0);
                }
            }
        }
    }

    SumProbe probe;
#pragma unroll
    for (int m = 0; m < MTW; m++) {
        const int o = (mt0 + m) * 16 + (lane >> 4) * 4;
        f32x4 sc = {0.f, 0.f, 0.f, 0.f};
        if (o < cstride) sc = *(const f32x4 *)(wscale + o);
#pragma unroll
        for (int t = 0; t < NTW; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                probe.scaled(acc[m][t][r]);
                acc[m][t][r] *= sc[r];
                probe.sum(acc[m][t][r]);
            }
    }
    if (__builtin_amdgcn_ballot_w64(probe.again())) {
#pragma unroll
        for (int m = 0; m < MTW; m++)
#pragma unroll
            for (int t = 0; t < NTW; t++) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        // (The empty asm keeps what is formed here out of the main loop's
        // registers.)
        int id = threadIdx.x;
        asm volatile("" : "+v"(id));
        const int l = id & 63, w2 = id >> 6;
        const int m0 = (blockIdx.y * 2 + (w2 & 1)) * MTW;
#pragma unroll 1
        for (int k = 0; k < steps * 8; k++) {
            // Four channels of a tap, one a lane group.
            const int s = k >> 3, c32 = (k & 7) * 4 + (l >> 4);
            const int chunk = s / FF, tap = s % FF, c = chunk * 32 + c32;
            float av[MTW], bv[NTW];
#pragma unroll
            for (int m = 0; m < MTW; m++) {
                const int at =
                    (m0 + m < mtiles ? m0 + m : mtiles - 1) * 64 + (l & 15) +
                    16 * (c32 >> 3);
                av[m] = wplain[((size_t)s * mtiles * 64 + at) * 8 + (c32 & 7)];
            }
#pragma unroll
            for (int t = 0; t < NTW; t++) {
                // (Columns past the band: any values, never stored.)
                const int j = ((w2 >> 1) * NTW + t) * 16 + (l & 15);
                const int y = y0 + j / kS + tap / F - F / 2;
                const int x = j % kS + tap % F - F / 2;
                const bool on = y >= 0 && y < kS && x >= 0 && x < kS;
                bv[t] = 0.f;
                if (NB == 1) {
                    if (on && c < cin)
                        bv[t] = (float)((const uint8_t *)
                                            in)[((size_t)board * cin + c) * kP +
                                                y * kS + x];
                } else if (on) {
                    bv[t] = ((const float *)in)[((size_t)board * kP + y * kS +
                                                 x) * (chunks * 32) + c];
                }
            }
#pragma unroll
            for (int m = 0; m < MTW; m++)
#pragma unroll
                for (int t = 0; t < NTW; t++)
                    acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                        av[m], bv[t], acc[m][t], 0, 0, 0);
        }
    }

    // D layout of 16x16 MFMA: lane holds rows 4*(lane/16)+r of column
    // lane%16: four channels of a pixel.
#pragma unroll
    for (int m = 0; m < MTW; m++) {
        const int o = (mt0 + m) * 16 + (lane >> 4) * 4;
        if (o >= cstride) continue;
        float bo[4], bm[4], ba[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const bool on = o + r < cout;
            bo[r] = on ? bias[o + r] : 0.f;
            bm[r] = on && epi.bn_mean ? epi.bn_mean[o + r] : 0.f;
            ba[r] = on && epi.bn_mean ? epi.bn_inv_std[o + r] : 1.f;
        }
#pragma unroll
        for (int t = 0; t < NTW; t++) {
            if (pix[t] < 0) continue;
            f32x4 v;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                v[r] = activate(acc[m][t][r] + bo[r], epi.act);
                // Network.cpp:445: scale_stddiv * (in - mean).
                if (epi.bn_mean) v[r] = ba[r] * (v[r] - bm[r]);
                if (o + r >= cout) v[r] = 0.f;
            }
            *(f32x4 *)(out + ((size_t)board * kP + pix[t]) * cstride + o) = v;
        }
    }
}

// ---- 1-channel head convs -------------------------------------------------
// The 3x3 conv to one channel as a product with the nine taps as rows:
// d[tap][p] = sum_c w[tap][c] x[p][c] (split as above, 16 rows of which nine
// are used), then out[p] = sum_tap d[tap][p shifted by the tap]. Every input
// value is read once, straight into an operand. Weights: [chunk][part]
// [lane][8], lane = tap + 16 * channel group, over the conv's scale. Where a
// sum is not finite or very small FP32 products take its place, as in
// conv_split.
constexpr int kHeadThreads = 512;
constexpr int kHeadPix = 368;  // 23 column tiles

// The activated conv of one board into s_out[0..361).
__device__ __forceinline__ void head_split(const float *__restrict__ src,
                                           const bf16x8 *__restrict__ w,
                                           const float *__restrict__ wscale,
                                           const float *__restrict__ wplain,
                                           float bias, int cin, int act,
                                           float (*d)[kHeadPix],
                                           float *s_out) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int chunks = (cin + 31) / 32;
    SumProbe probe;
    for (int t = wave; t < kHeadPix / 16; t += kHeadThreads / 64) {
        const int p = t * 16 + (lane & 15);
        const f32x4 *x = (const f32x4 *)(src + (size_t)(p < kP ? p : kP - 1) *
                                                   chunks * 32) +
                         (lane >> 4) * 2;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
        for (int c = 0; c < chunks; c++) {
            const f32x4 lo = x[c * 8], hi = x[c * 8 + 1];
            float v[8];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v[e] = lo[e];
                v[4 + e] = hi[e];
            }
            bf16x8 b[3], a[3];
            split3(v, b);
#pragma unroll
            for (int q = 0; q < 3; q++) a[q] = w[(c * 3 + q) * 64 + lane];
            acc = Op<__bf16>::mfma(a[0], b[2], acc);
            acc = Op<__bf16>::mfma(a[2], b[0], acc);
            acc = Op<__bf16>::mfma(a[1], b[1], acc);
            acc = Op<__bf16>::mfma(a[0], b[1], acc);
            acc = Op<__bf16>::mfma(a[1], b[0], acc);
            acc = Op<__bf16>::mfma(a[0], b[0], acc);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            if ((lane >> 4) * 4 + r < 9) d[(lane >> 4) * 4 + r][p] = acc[r];
            probe.scaled(acc[r]);
            probe.sum(acc[r]);
        }
    }
    const bool again = __syncthreads_or(probe.again());
    for (int p = tid; p < kP; p += kHeadThreads) {
        const int y = p / kS, x = p % kS;
        float v = 0.0f;
#pragma unroll
        for (int tap = 0; tap < 9; tap++) {
            const int yy = y + tap / 3 - 1, xx = x + tap % 3 - 1;
            if (yy >= 0 && yy < kS && xx >= 0 && xx < kS)
                v += d[tap][yy * kS + xx];
        }
        v *= wscale[0];
        if (again || !isfinite(v)) {
            v = 0.0f;
            for (int c = 0; c < cin; c++)
                for (int tap = 0; tap < 9; tap++) {
                    const int yy = y + tap / 3 - 1, xx = x + tap % 3 - 1;
                    const bool on = yy >= 0 && yy < kS && xx >= 0 && xx < kS;
                    v += wplain[c * 9 + tap] *
                         (on ? src[(size_t)(yy * kS + xx) * chunks * 32 + c]
                             : 0.f);
                }
        }
        s_out[p] = activate(v + bias, act);
    }
    __syncthreads();
}

__device__ float block_reduce(float v, bool is_max, float *s_red) {
    for (int off = 32; off > 0; off >>= 1) {
        const float o = __shfl_xor(v, off, 64);
        v = is_max ? fmaxf(v, o) : v + o;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) s_red[wave] = v;
    __syncthreads();
    float r = s_red[0];
    for (int i = 1; i < kHeadThreads / 64; i++)
        r = is_max ? fmaxf(r, s_red[i]) : r + s_red[i];
    return r;
}

__global__ __launch_bounds__(kHeadThreads) void policy_head_f32_kernel(
    const float *__restrict__ in, const bf16x8 *__restrict__ w,
    const float *__restrict__ wscale, const float *__restrict__ wplain,
    const float *__restrict__ b, float *__restrict__ raw,
    float *__restrict__ out, int cin, float temperature, int act) {
    __shared__ float d[9][kHeadPix];
    __shared__ float s_logit[kP];
    __shared__ float s_red[kHeadThreads / 64];
    const int board = blockIdx.x, p = threadIdx.x;
    head_split(in + (size_t)board * kP * ((cin + 31) / 32 * 32), w, wscale,
               wplain, b[0], cin, act, d, s_logit);
    // Network::softmax (Network.cpp:450-469): exp(x/T - max/T) / sum.
    const float v = p < kP ? s_logit[p] : -INFINITY;
    const float alpha = block_reduce(v, true, s_red) / temperature;
    const float e = p < kP ? expf(v / temperature - alpha) : 0.0f;
    const float sum = block_reduce(e, false, s_red);
    if (p >= kP) return;
    if (raw) raw[(size_t)board * kP + p] = v;
    if (out) out[(size_t)board * kP + p] = e / sum;
}

// Last 1-channel conv + activation of the value net, written to h0
// [n][361] for value_fc_head.
__global__ __launch_bounds__(kHeadThreads) void value_headconv_f32_kernel(
    const float *__restrict__ in, const bf16x8 *__restrict__ w,
    const float *__restrict__ wscale, const float *__restrict__ wplain,
    const float *__restrict__ b, float *__restrict__ h0, int cin, int act) {
    __shared__ float d[9][kHeadPix];
    __shared__ float s_h0[kP];
    const int board = blockIdx.x, p = threadIdx.x;
    head_split(in + (size_t)board * kP * ((cin + 31) / 32 * 32), w, wscale,
               wplain, b[0], cin, act, d, s_h0);
    if (p < kP) h0[(size_t)board * kP + p] = s_h0[p];
}

// Batched inner-product head of the value net (Network.cpp:733-736):
// hidden = ELU(W1 h0 + b1), v = w2 . hidden + b2, out = (1 + tanh v) / 2.
// A workgroup takes kFcBoards boards so that every W1 element from L2 is
// used kFcBoards times. Bound: the latency of those reads (370 KB through
// each CU). A lane forms four hidden units, the eight waves share the inputs
// (every eighth each), and eight rows of W1 are on the way per wave: 64 KB
// in flight on a CU, where a unit per thread had 8 KB: 22.6 / 22.8 -> 9.7 /
// 10.9 us at 16 / 1024 boards (kernel trace). Four boards per workgroup keep a batch of 1024 on 256
// workgroups (one per CU).
constexpr int kFcBoards = 4, kFcThreads = 512;

// VEC: H is a multiple of 4 (rows of W1 are read 16 bytes at a time).
template <bool VEC>
__global__ __launch_bounds__(kFcThreads) void value_fc_kernel(
    const float *__restrict__ h0, const float *__restrict__ w1t,
    const float *__restrict__ b1, const float *__restrict__ w2,
    const float *__restrict__ b2, float *__restrict__ raw,
    float *__restrict__ out, int n, int P, int H,
    const int *__restrict__ n_dev) {
    constexpr int W = kFcThreads / 64;
    __shared__ f32x4 s_h[kMaxSide * kMaxSide];  // [input] (boards)
    __shared__ float s_part[W][kFcBoards][256];
    __shared__ float s_red[kFcBoards][W];
    // A replayed graph sizes its grid for the bucket; the batch's board
    // count is then read from device memory.
    if (n_dev) n = min(n, *n_dev);
    const int b0 = blockIdx.x * kFcBoards, tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (b0 >= n) return;
    const int nb = min(kFcBoards, n - b0);
    for (int i = tid; i < P; i += kFcThreads) {
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int bb = 0; bb < kFcBoards; bb++)
            if (bb < nb) v[bb] = h0[(size_t)(b0 + bb) * P + i];
        s_h[i] = v;
    }
    __syncthreads();
    float part[kFcBoards];
#pragma unroll
    for (int bb = 0; bb < kFcBoards; bb++) part[bb] = 0.0f;
    for (int j = 0; j < H; j += 256) {
        const int o = j + lane * 4;
        f32x4 acc[kFcBoards];
#pragma unroll
        for (int bb = 0; bb < kFcBoards; bb++) acc[bb] = f32x4{0.f, 0.f, 0.f, 0.f};
        // Row i0 + u W of W1 (past the last input the last row, not used: its
        // weights times zeros would be NaN where one is infinite).
        f32x4 wv[8];
        auto row_at = [&](int i) {
            const float *row = w1t + (size_t)min(i, P - 1) * H;
            f32x4 v;
            if (VEC) {
                v = *(const f32x4 *)(row + min(o, H - 4));
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++) v[r] = row[min(o + r, H - 1)];
            }
            return v;
        };
#pragma unroll
        for (int u = 0; u < 8; u++) wv[u] = row_at(wave + u * W);
        auto add = [&](const f32x4 &w, const f32x4 &h) {
#pragma unroll
            for (int bb = 0; bb < kFcBoards; bb++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[bb][r] += w[r] * h[bb];
        };
        int i0 = wave;
        for (; i0 + 7 * W < P; i0 += 8 * W) {
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const f32x4 h = s_h[i0 + u * W], w = wv[u];
                wv[u] = row_at(i0 + (u + 8) * W);
                add(w, h);
            }
        }
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (i0 + u * W < P) add(wv[u], s_h[i0 + u * W]);
        __syncthreads();
#pragma unroll
        for (int bb = 0; bb < kFcBoards; bb++)
            *(f32x4 *)&s_part[wave][bb][lane * 4] = acc[bb];
        __syncthreads();
        if (tid < 256 && j + tid < H) {
            const float bo = b1[j + tid], wo = w2[j + tid];
#pragma unroll
            for (int bb = 0; bb < kFcBoards; bb++) {
                float v = s_part[0][bb][tid];
#pragma unroll
                for (int q = 1; q < W; q++) v += s_part[q][bb][tid];
                part[bb] += wo * elu(v + bo);
            }
        }
    }
#pragma unroll
    for (int bb = 0; bb < kFcBoards; bb++) {
        float v = part[bb];
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
        if (lane == 0) s_red[bb][wave] = v;
    }
    __syncthreads();
    if (tid < nb) {
        float v = b2[0];
        for (int q = 0; q < W; q++) v += s_red[tid][q];
        if (raw) raw[b0 + tid] = v;
        if (out) out[b0 + tid] = (1.0f + tanhf(v)) / 2.0f;
    }
}

template <int F, int NB, int MTW, int NTW>
hipError_t launch(const void *in, const SplitWeights &w, const float *bias,
                  float *out, int n, int cin, int cout,
                  const ConvEpilogue &epi, hipStream_t stream) {
    constexpr int BANDS = NTW == 6 ? 2 : 4;
    const int mtiles = (cout + 15) / 16;
    const dim3 grid(n * BANDS, (mtiles + 2 * MTW - 1) / (2 * MTW));
    hipLaunchKernelGGL((conv_split<F, NB, MTW, NTW>), grid, dim3(kThreads), 0,
                       stream, in, reinterpret_cast<const bf16x8 *>(w.parts),
                       w.scale, w.plain, bias, out, cin, f32_chunks(cin), cout,
                       f32_stride(cout), mtiles, epi);
    return hipGetLastError();
}

// The piece of a conv that a workgroup takes, by a model of the time: a
// workgroup costs its MFMAs (MTW x NTW) and its staging (2, or 4 for ten
// rows), a CU's share is ceil(workgroups / 256) of them, and one workgroup
// alone on a CU runs 1.6 times as long as its share of a full one. On a tie
// the larger piece (it stages each input value for more outputs). The model
// holds within 10% over n = 32 .. 256 (2.05 us a unit for 128 -> 128: 12
// convs at n = 64 take 458 us with one m-tile and five rows a wave, 564 with
// four; at n = 256 1339 us with four and ten, 1416 with four and five).
template <int F, int NB>
hipError_t launch_conv(const void *in, const SplitWeights &w, const float *bias,
                       float *out, int n, int cin, int cout,
                       const ConvEpilogue &epi, hipStream_t stream) {
    const int mtiles = (cout + 15) / 16;
    int mtw = 4;
    bool big = true;
    double best = 0.0;
    for (int k = 4; k >= 1; k--)
        for (int rows10 = 1; rows10 >= 0; rows10--) {
            const long long blocks = (mtiles + 2 * k - 1) / (2 * k);
            const long long wgs = n * (rows10 ? 2LL : 4LL) * blocks;
            const double q = (double)((wgs + 255) / 256);
            const double t = (q < 2 ? 1.6 : q) *
                             (k * (rows10 ? 6 : 3) + (rows10 ? 4 : 2));
            if (best == 0.0 || t < best) {
                best = t;
                mtw = k;
                big = rows10;
            }
        }
    auto go = [&](auto m) {
        constexpr int M = decltype(m)::value;
        return big ? launch<F, NB, M, 6>(in, w, bias, out, n, cin, cout, epi,
                                         stream)
                   : launch<F, NB, M, 3>(in, w, bias, out, n, cin, cout, epi,
                                         stream);
    };
    switch (mtw) {
    case 1: return go(std::integral_constant<int, 1>());
    case 2: return go(std::integral_constant<int, 2>());
    case 3: return go(std::integral_constant<int, 3>());
    default: return go(std::integral_constant<int, 4>());
    }
}

bool act_ok(int act) {
    return act == kActElu || act == kActRelu || act == kActNone;
}

}  // namespace

hipError_t conv_f32(int filter, bool u8_input, const void *in,
                    const SplitWeights &w, const float *bias, float *out,
                    int n, int cin, int cout, const ConvEpilogue &epi,
                    hipStream_t stream) {
    if (n <= 0 || cin < 1 || cout < 1 || !act_ok(epi.act) ||
        (epi.bn_mean && !epi.bn_inv_std))
        return hipErrorInvalidValue;
    if (filter == 3)
        return u8_input ? launch_conv<3, 1>(in, w, bias, out, n, cin, cout,
                                            epi, stream)
                        : launch_conv<3, 3>(in, w, bias, out, n, cin, cout,
                                            epi, stream);
    if (filter == 5)
        return u8_input ? launch_conv<5, 1>(in, w, bias, out, n, cin, cout,
                                            epi, stream)
                        : launch_conv<5, 3>(in, w, bias, out, n, cin, cout,
                                            epi, stream);
    return hipErrorInvalidValue;
}

hipError_t policy_head_f32(const float *in, const SplitWeights &w,
                           const float *b, float *raw, float *out, int n,
                           int cin, float temperature, int act,
                           hipStream_t stream) {
    if (n <= 0 || cin < 1 || !act_ok(act)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(policy_head_f32_kernel, dim3(n), dim3(kHeadThreads), 0,
                       stream, in, reinterpret_cast<const bf16x8 *>(w.parts),
                       w.scale, w.plain, b, raw, out, cin, temperature, act);
    return hipGetLastError();
}

hipError_t value_headconv_f32(const float *in, const SplitWeights &w,
                              const float *b, float *h0, int n, int cin,
                              int act, hipStream_t stream) {
    if (n <= 0 || cin < 1 || !act_ok(act)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(value_headconv_f32_kernel, dim3(n), dim3(kHeadThreads),
                       0, stream, in, reinterpret_cast<const bf16x8 *>(w.parts),
                       w.scale, w.plain, b, h0, cin, act);
    return hipGetLastError();
}

hipError_t value_fc_head(const float *h0, const float *fc1_wt,
                         const float *fc1_b, const float *fc2_w,
                         const float *fc2_b, float *raw, float *out, int n,
                         int P, int hidden, hipStream_t stream,
                         const int *n_dev) {
    if (n <= 0) return hipSuccess;
    if (P < 1 || P > kMaxSide * kMaxSide || hidden < 1)
        return hipErrorInvalidValue;
    const int grid = (n + kFcBoards - 1) / kFcBoards;
    const auto fn =
        hidden % 4 == 0 ? value_fc_kernel<true> : value_fc_kernel<false>;
    hipLaunchKernelGGL(fn, dim3(grid), dim3(kFcThreads), 0, stream, h0, fc1_wt,
                       fc1_b, fc2_w, fc2_b, raw, out, n, P, hidden, n_dev);
    return hipGetLastError();
}

}  // namespace lz
