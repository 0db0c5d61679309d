// surrogate.hip — training and inference kernels of the learned playout
// surrogate (network in lz_surrogate.h).
//
// Forward — sg_fwd
//   The whole network for one board per workgroup in one launch: the board
//   stays in LDS as a zero-haloed BF16 HWC tile (lz_conv_tile.h's layout)
//   through all 13 convs, each an implicit GEMM on
//   v_mfma_f32_16x16x32_bf16 with packed weights from L2 (sg_pack), then
//   the FP32 head. Every conv output also goes to its map in HBM (the
//   backward pass and read_map take them from there) and nothing is read
//   back: residuals stay in the registers of the lanes that formed them. The
//   FP32 epilogue adds bias and residual and applies ELU.
//   Bound: MFMA and its operand reads from n = 512 up (333 MFLOP a board),
//   with the maps' stores (0.6 MB a board) beside them; one conv's latency,
//   13 times, below one board per CU. At n = 4096: 1.32 ms (1.03 PFLOP/s;
//   1.09 ms with the stores taken out), against 3.37 ms for one launch per
//   conv with its input staged from HBM each time. Residuals read back from
//   HBM instead of kept in registers cost 0.7 ms of the 4096, stores of 8
//   bytes straight from the accumulators 0.4 ms.
//
// Backward-data — sg_conv
//   One workgroup per board, 4 waves. The gradient map is staged into LDS as
//   a 21x21 BF16 HWC tile with a zero halo (pixel stride 72 staggers pixels
//   across banks). Wave w owns pixel tiles w, w+4, ... (6 or 5 of the 23)
//   for all 64 output channels. dX = conv(dY; W') with
//   W'[c][o][tap] = W[o][c][8 - tap] (taps flipped), packed by sg_pack; the
//   epilogue adds the skip's gradient, multiplies by ELU's derivative taken
//   from the stored forward activation, and stores BF16 quads.
//
// Weight gradient — sg_wgrad
//   dW[o][c][tap] = sum over boards and pixels of e[p][o] x[p + tap][c]:
//   a GEMM whose reduction runs over pixels, so both operands are staged
//   transposed (channel rows, pixel columns) in LDS. Pixels are indexed in
//   a 19x21 frame (two zero columns per row, 399 -> 416 = 13 k-steps), and
//   the input is staged already shifted by the workgroup's tap, so every
//   fragment is one aligned 16-byte ds_read. Grid = 9 taps x board chunks;
//   each workgroup writes its FP32 partial, and a second kernel sums the
//   chunks in a fixed order (deterministic) into OIHW.
//
// Head (ELU activations), loss, Adam: FP32, small kernels (the head is
// 0.2% of the FLOPs).
#include "lz_conv_tile.h"
#include "lz_surrogate.h"

namespace lz {
namespace sg {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

constexpr int S = kSide, P = kP;
constexpr int HS = S + 2, HP = HS * HS;   // halo frame 21 x 21
constexpr int NT = (P + 15) / 16;         // 23 pixel tiles
constexpr int KF = 416;                   // 19 x 21 frame, 13 k-steps of 32
constexpr int KFP = KF + 8;               // LDS row pitch (bank stagger)
constexpr int kThreads = 256;
constexpr int kMaxChunks = 64;
// Batches of at most this many boards (one per CU) use eight waves a board:
// 95 us up to n = 200 and 102 at 256, against 122-124 with four; from 257 on
// a CU holds two boards and four waves each are faster (152 against 173 us
// at 257, 332 against 354 at 1024).
constexpr int kWideBoards = 256;

__device__ inline f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// The activation of every layer: ELU, as in the reference nets
// (Network.cpp:387-392). With ReLU, training runs collapsed to a constant
// output (every unit of a layer switched off); ELU keeps a gradient
// everywhere.
__device__ inline float elu(float v) { return v > 0.f ? v : expf(v) - 1.f; }
// d ELU / d v expressed through the output a = ELU(v).
__device__ inline float elu_grad(float a) { return a > 0.f ? 1.f : a + 1.f; }

__device__ inline float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

int chunks_for(int n) { return n < kMaxChunks ? n : kMaxChunks; }

// ---- weight packing --------------------------------------------------------
// All convs' MFMA A-operands, forward and (64 -> 64 only) backward-data, in
// one launch: 25 launches of 9 us of tiny work each were 0.12 ms of a
// training step. Blocks of the forward weights first, layer by layer, then
// the backward ones; a thread forms one fragment's 8 values.
constexpr int kPack0 = 9 * 32 * kCh / 8 / kThreads;   // blocks of layer 0
constexpr int kPackL = 9 * kCh * kCh / 8 / kThreads;  // of any other
static_assert(kPack0 * 8 * kThreads == 9 * 32 * kCh &&
                  kPackL * 8 * kThreads == 9 * kCh * kCh, "whole blocks");

__global__ __launch_bounds__(kThreads) void sg_pack(PackArgs a) {
    int blk = blockIdx.x, l = 0, cin = 32;
    bool bwd = false;
    if (blk >= kPack0) {
        blk -= kPack0;
        l = 1 + blk / kPackL;
        blk %= kPackL;
        cin = kCh;
        if (l >= kNConv) {
            l -= kNConv - 1;
            bwd = true;
        }
    }
    const float *w = a.w[l];
    const int i = blk * kThreads + threadIdx.x;
    const int lane = i & 63, mt = (i >> 6) & 3, ks = i >> 8;
    const int k = ks * 32 + (lane >> 4) * 8;
    const int row = mt * 16 + (lane & 15);
    const int tap = k / cin, c = k % cin;  // 8 values: one tap
    bf16x8 v;
#pragma unroll
    for (int e = 0; e < 8; e++)
        // Backward: row = forward input channel, c = forward output channel.
        v[e] = (__bf16)(bwd ? w[((c + e) * kCh + row) * 9 + (8 - tap)]
                            : w[(row * cin + c + e) * 9 + tap]);
    reinterpret_cast<bf16x8 *>(bwd ? a.wb[l] : a.wf[l])[i] = v;
}

// ---- the forward pass ---------------------------------------------------------
constexpr int kPS = kCh + 16;                    // pixel stride, trunk tile
constexpr int kInPS = 48;                        // of the 32 input planes
constexpr int kRP = HS * kPS + row_pad(kPS, 2);  // row pitch
constexpr int kInRP = HS * kInPS + row_pad(kInPS, 2);
constexpr int kTile = HS * kRP;
static_assert(kInRP <= kRP && kTile % 8 == 0, "the input fits the tile");

// The lane's pixel offsets in its wave's column tiles: window origins in the
// trunk tile (pb) and the pixel index (pix, -1 past the board).
__device__ __forceinline__ void sg_geom(int wn, int lane, int (&pb)[kNT],
                                        int (&pix)[kNT]) {
#pragma unroll
    for (int t = 0; t < kNT; t++) {
        const int j = (wn * kNT + t) * 16 + (lane & 15);
        pix[t] = j < P ? j : -1;
        // A lane past the board reads the pixel a multiple of 16 before it.
        const int jj = j < P ? j : j - ((j - P) / 16 + 1) * 16;
        pb[t] = (jj / S) * kRP + (jj % S) * kPS;
    }
}

// Epilogue of a forward conv (bias in the accumulators): + residual, ELU,
// BF16 into the tile. acc's lane holds four consecutive channels of one
// pixel per fragment. keep: the lane's outputs of the last even conv, which
// are the residual of an even conv (kRes) and are replaced by its outputs
// (kKeep).
template <bool kRes, bool kKeep, int MTW>
__device__ __forceinline__ void sg_store_fwd(__bf16 *tile,
                                             const f32x4 (&acc)[MTW][kNT],
                                             bf16x4 (&keep)[MTW][kNT],
                                             int mt0, const int (&pb)[kNT],
                                             const int (&pix)[kNT], int lane) {
    const int g4 = (lane >> 4) * 4;
#pragma unroll
    for (int m = 0; m < MTW; m++) {
        const int o = (mt0 + m) * 16 + g4;
#pragma unroll
        for (int t = 0; t < kNT; t++) {
            bf16x4 v;
#pragma unroll
            for (int r = 0; r < 4; r++)
                v[r] = (__bf16)elu_operand(
                    kRes ? acc[m][t][r] + (float)keep[m][t][r] : acc[m][t][r]);
            if (kKeep) keep[m][t] = v;
            if (pix[t] >= 0)
                *(bf16x4 *)(tile + pb[t] + kRP + kPS + o) = v;
        }
    }
}

// Copies the tile's board to its map in HBM, 16 bytes a lane (T threads).
// kStream: past the caches, for maps that no kernel of the call reads. Four
// stores at a time where registers are short (T = 256).
template <int T, bool kStream>
__device__ __forceinline__ void sg_copy_out(const __bf16 *tile, __bf16 *map,
                                            int tid) {
    constexpr int kUnroll = T > kThreads ? 6 : 4;
#pragma unroll kUnroll
    for (int k = 0; k < (P * 8 + T - 1) / T; k++) {
        const int i = tid + k * T, p = i >> 3;
        if (i >= P * 8) break;
        const bf16x8 v = *(const bf16x8 *)(tile + (p / S + 1) * kRP +
                                           (p % S + 1) * kPS + (i & 7) * 8);
        if (kStream)
            __builtin_nontemporal_store(v, (bf16x8 *)(map + i * 8));
        else
            *(bf16x8 *)(map + i * 8) = v;
    }
}

// kWM waves split the output channels, four the pixels. kWM = 1: two
// workgroups (75 KB of LDS each) per CU; kWM = 2 halves a board's latency
// where a CU holds one board only.
template <int kWM, bool kStream>
__global__ __launch_bounds__(kWM * kThreads, 2) void sg_fwd(
    const uint8_t *__restrict__ planes, FwdArgs a, uint16_t *act,
    size_t map_elems, const float *__restrict__ hp,
    float *__restrict__ s_out, float *__restrict__ f_out,
    float *__restrict__ t_out, float *__restrict__ win) {
    constexpr int T = kWM * kThreads, W = kWM * 4;
    constexpr int MT = kCh / 16, MTW = MT / kWM;
    __shared__ __attribute__((aligned(16))) __bf16 tile[kTile];
    __shared__ float s[P];
    __shared__ float f[kHid];
    const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int mt0 = (w / kWN) * MTW;
    const bf16x8 zero8 = {};
    __bf16 *maps = (__bf16 *)act + (size_t)b * P * kCh;

    // The planes with a zero halo: a thread takes 8 planes of a point.
    const uint8_t *pl = planes + (size_t)b * 32 * P;
    for (int i = tid; i < HP * 4; i += T) {
        const int hpx = i % HP, c8 = i / HP;
        const int y = hpx / HS - 1, x = hpx % HS - 1;
        bf16x8 v = zero8;
        if (y >= 0 && y < S && x >= 0 && x < S) {
#pragma unroll
            for (int e = 0; e < 8; e++)
                v[e] = (__bf16)(float)pl[(c8 * 8 + e) * P + y * S + x];
        }
        *(bf16x8 *)(tile + (y + 1) * kInRP + (x + 1) * kInPS + c8 * 8) = v;
    }
    int pb[kNT], pix[kNT];
    sg_geom(w % kWN, lane, pb, pix);
    __syncthreads();
    bf16x4 keep[MTW][kNT];
    {
        f32x4 acc[MTW][kNT];
        int pbi[kNT];
#pragma unroll
        for (int t = 0; t < kNT; t++)
            pbi[t] = pb[t] / kRP * kInRP + pb[t] % kRP / kPS * kInPS;
        conv_tile<__bf16, 3, 32, MT, MTW, kInPS>(
            tile, (const bf16x8 *)a.w[0], acc, pbi, kInRP, mt0, lane, a.b[0]);
        __syncthreads();
        for (int i = tid * 8; i < kTile; i += T * 8)
            *(bf16x8 *)(tile + i) = zero8;
        __syncthreads();
        sg_store_fwd<false, true, MTW>(tile, acc, keep, mt0, pb, pix, lane);
        __syncthreads();
    }
    // The map of a conv's input goes out between its MFMAs and its epilogue:
    // loads and stores retire in order, so stores ahead of a conv would
    // hold up its weight loads, and here the epilogue's math covers them.
    for (int l = 1; l < kNConv; l += 2) {
        f32x4 acc[MTW][kNT];
        conv_tile<__bf16, 3, kCh, MT, MTW, kPS>(
            tile, (const bf16x8 *)a.w[l], acc, pb, kRP, mt0, lane, a.b[l]);
        sg_copy_out<T, kStream>(tile, maps + (l - 1) * map_elems, tid);
        __syncthreads();
        sg_store_fwd<false, false, MTW>(tile, acc, keep, mt0, pb, pix, lane);
        __syncthreads();
        conv_tile<__bf16, 3, kCh, MT, MTW, kPS>(
            tile, (const bf16x8 *)a.w[l + 1], acc, pb, kRP, mt0, lane,
            a.b[l + 1]);
        sg_copy_out<T, kStream>(tile, maps + l * map_elems, tid);
        __syncthreads();
        sg_store_fwd<true, true, MTW>(tile, acc, keep, mt0, pb, pix, lane);
        __syncthreads();
    }
    sg_copy_out<T, kStream>(tile, maps + (kNConv - 1) * map_elems, tid);

    // Head, FP32. hp: wh[64], bh, F1[64][361], c1[64], F2[64], c2.
    const float *wh = hp, *F1 = hp + kCh + 1;
    const float *c1 = F1 + kHid * P, *F2 = c1 + kHid;
    for (int p = tid; p < P; p += T) {
        const bf16x8 *hv = (const bf16x8 *)(tile + (p / S + 1) * kRP +
                                            (p % S + 1) * kPS);
        float d = hp[kCh];
#pragma unroll
        for (int c8 = 0; c8 < 8; c8++) {
            const bf16x8 v = hv[c8];
#pragma unroll
            for (int k = 0; k < 8; k++) d += wh[c8 * 8 + k] * (float)v[k];
        }
        d = elu(d);
        s[p] = d;
        s_out[(size_t)b * P + p] = d;
    }
    __syncthreads();
    // A wave's kHid / W rows of F1 side by side: one wait for the loads of
    // all of them per 64 points.
    constexpr int J = kHid / W;
    float d[J];
#pragma unroll
    for (int j = 0; j < J; j++) d[j] = 0.f;
#pragma unroll
    for (int i = 0; i < (P + 63) / 64; i++) {
        const int p = i * 64 + lane;
        if (p < P) {
            const float sp = s[p];
#pragma unroll
            for (int j = 0; j < J; j++) d[j] += F1[(w * J + j) * P + p] * sp;
        }
    }
#pragma unroll
    for (int j = 0; j < J; j++) {
        const float v = wave_sum(d[j]);
        if (lane == j) {
            const float fj = elu(v + c1[w * J + j]);
            f[w * J + j] = fj;
            f_out[(size_t)b * kHid + w * J + j] = fj;
        }
    }
    __syncthreads();
    if (w == 0) {
        const float v = wave_sum(F2[lane] * f[lane]);
        if (lane == 0) {
            const float t = tanhf(v + F2[kHid]);
            t_out[b] = t;
            if (win) win[b] = 0.5f * (1.f + t);
        }
    }
}

// ---- backward-data convolution ------------------------------------------------
__global__ __launch_bounds__(kThreads, 2) void sg_conv(
    const __bf16 *__restrict__ in, const bf16x8 *__restrict__ wpk,
    const __bf16 *__restrict__ res, const __bf16 *__restrict__ mask,
    __bf16 *__restrict__ out) {
    constexpr int PS = kCh + 8;
    constexpr int C8 = kCh / 8;
    __shared__ __attribute__((aligned(16))) __bf16 tile[HP * PS];
    const int b = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;

    const bf16x8 zero8 = {};
    for (int i = tid; i < HP * C8; i += kThreads) {
        const int hp = i / C8, c8 = i % C8;
        const int hy = hp / HS, hx = hp % HS;
        if (hy == 0 || hy == HS - 1 || hx == 0 || hx == HS - 1)
            *(bf16x8 *)&tile[hp * PS + c8 * 8] = zero8;
    }
    const bf16x8 *src = (const bf16x8 *)in + (size_t)b * P * C8;
    for (int i = tid; i < P * C8; i += kThreads) {
        const int p = i / C8, c8 = i % C8;
        const int y = p / S, x = p % S;
        *(bf16x8 *)&tile[((y + 1) * HS + x + 1) * PS + c8 * 8] = src[i];
    }
    __syncthreads();

    int hp0[6];
#pragma unroll
    for (int jj = 0; jj < 6; jj++) {
        const int px = (w + 4 * jj) * 16 + (lane & 15);
        hp0[jj] = px < P ? (px / S + 1) * HS + px % S + 1 : -1;
    }
    f32x4 acc[6][4];
#pragma unroll
    for (int jj = 0; jj < 6; jj++)
#pragma unroll
        for (int mt = 0; mt < 4; mt++) acc[jj][mt] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int kq = (lane >> 4) * 8;
    constexpr int KS = 9 * kCh / 32;
    for (int ks = 0; ks < KS; ks++) {
        const int tap = (ks * 32) / kCh, c0 = (ks * 32) % kCh;
        const int off = (tap / 3 - 1) * HS + (tap % 3 - 1);
        bf16x8 a[4];
#pragma unroll
        for (int mt = 0; mt < 4; mt++) a[mt] = wpk[(ks * 4 + mt) * 64 + lane];
#pragma unroll
        for (int jj = 0; jj < 6; jj++) {
            if (w + 4 * jj >= NT) continue;
            const int hp = hp0[jj] >= 0 ? hp0[jj] + off : 0;
            const bf16x8 bv = *(const bf16x8 *)&tile[hp * PS + c0 + kq];
#pragma unroll
            for (int mt = 0; mt < 4; mt++) acc[jj][mt] = mfma(a[mt], bv, acc[jj][mt]);
        }
    }

    const int orow = (lane >> 4) * 4;
#pragma unroll
    for (int jj = 0; jj < 6; jj++) {
        const int px = (w + 4 * jj) * 16 + (lane & 15);
        if (w + 4 * jj >= NT || px >= P) continue;
#pragma unroll
        for (int mt = 0; mt < 4; mt++) {
            const int o = mt * 16 + orow;
            const size_t at = ((size_t)b * P + px) * kCh + o;
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = acc[jj][mt][r];
            if (res) {
                const bf16x4 rv = *(const bf16x4 *)(res + at);
#pragma unroll
                for (int r = 0; r < 4; r++) v[r] += (float)rv[r];
            }
            const bf16x4 mv = *(const bf16x4 *)(mask + at);
            bf16x4 ov;
#pragma unroll
            for (int r = 0; r < 4; r++)
                ov[r] = (__bf16)(v[r] * elu_grad((float)mv[r]));
            *(bf16x4 *)(out + at) = ov;
        }
    }
}

// ---- weight gradient -----------------------------------------------------------
template <int CIN>
__global__ __launch_bounds__(kThreads, 1) void sg_wgrad(
    const void *__restrict__ in, const __bf16 *__restrict__ e,
    float *__restrict__ part, int n, int bpc) {
    __shared__ __attribute__((aligned(16))) __bf16 eT[kCh * KFP];
    __shared__ __attribute__((aligned(16))) __bf16 xT[CIN * KFP];
    constexpr int NTC = CIN / 16;
    const int tap = blockIdx.x % 9, chunk = blockIdx.x / 9;
    const int dy = tap / 3 - 1, dx = tap % 3 - 1;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int b0 = chunk * bpc;
    const int b1 = b0 + bpc < n ? b0 + bpc : n;

    f32x4 acc[NTC];
#pragma unroll
    for (int nt = 0; nt < NTC; nt++) acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float dbacc = 0.f;

    for (int b = b0; b < b1; b++) {
        // e^T[o][p'], p' = y * 21 + x in the 19 x 21 frame.
        for (int i = tid; i < KF * 8; i += kThreads) {
            const int pp = i >> 3, o8 = i & 7;
            const int y = pp / HS, x = pp % HS;
            bf16x8 v = {};
            if (y < S && x < S)
                v = *(const bf16x8 *)(e + ((size_t)b * P + y * S + x) * kCh + o8 * 8);
#pragma unroll
            for (int k = 0; k < 8; k++) eT[(o8 * 8 + k) * KFP + pp] = v[k];
        }
        // x^T[c][p'] = input at (y + dy, x + dx), zero off the board.
        if (CIN == 32) {
            const uint8_t *pl = (const uint8_t *)in + (size_t)b * 32 * P;
            for (int i = tid; i < 32 * KF; i += kThreads) {
                const int c = i / KF, pp = i % KF;
                const int y = pp / HS + dy, x = pp % HS + dx;
                float v = 0.f;
                if (pp / HS < S && pp % HS < S && y >= 0 && y < S && x >= 0 && x < S)
                    v = (float)pl[c * P + y * S + x];
                xT[c * KFP + pp] = (__bf16)v;
            }
        } else {
            for (int i = tid; i < KF * 8; i += kThreads) {
                const int pp = i >> 3, c8 = i & 7;
                const int y = pp / HS + dy, x = pp % HS + dx;
                bf16x8 v = {};
                if (pp / HS < S && pp % HS < S && y >= 0 && y < S && x >= 0 && x < S)
                    v = *(const bf16x8 *)((const __bf16 *)in +
                                          ((size_t)b * P + y * S + x) * kCh + c8 * 8);
#pragma unroll
                for (int k = 0; k < 8; k++) xT[(c8 * 8 + k) * KFP + pp] = v[k];
            }
        }
        __syncthreads();
        for (int ks = 0; ks < KF / 32; ks++) {
            const int k0 = ks * 32 + (lane >> 4) * 8;
            const bf16x8 a = *(const bf16x8 *)&eT[(w * 16 + (lane & 15)) * KFP + k0];
#pragma unroll
            for (int nt = 0; nt < NTC; nt++) {
                const bf16x8 bv = *(const bf16x8 *)&xT[(nt * 16 + (lane & 15)) * KFP + k0];
                acc[nt] = mfma(a, bv, acc[nt]);
            }
        }
        if (tap == 4 && tid < kCh) {
            float s = 0.f;
            for (int pp = 0; pp < KF; pp++) s += (float)eT[tid * KFP + pp];
            dbacc += s;
        }
        __syncthreads();
    }
    // Partial layout: [chunk][tap][o][c], then [chunk][o] bias sums after
    // all chunks' weight partials.
    float *dst = part + ((size_t)chunk * 9 + tap) * kCh * CIN;
#pragma unroll
    for (int nt = 0; nt < NTC; nt++)
#pragma unroll
        for (int r = 0; r < 4; r++)
            dst[(w * 16 + (lane >> 4) * 4 + r) * CIN + nt * 16 + (lane & 15)] = acc[nt][r];
    if (tap == 4 && tid < kCh) {
        const int nch = gridDim.x / 9;
        part[(size_t)nch * 9 * kCh * CIN + chunk * kCh + tid] = dbacc;
    }
}

template <int CIN>
__global__ __launch_bounds__(kThreads) void sg_wgrad_reduce(
    const float *__restrict__ part, int nch, float *__restrict__ gW,
    float *__restrict__ gb) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    constexpr int N = 9 * kCh * CIN;
    if (i < N) {
        float s = 0.f;
        for (int ch = 0; ch < nch; ch++) s += part[(size_t)ch * N + i];
        const int tap = i / (kCh * CIN), o = (i / CIN) % kCh, c = i % CIN;
        gW[(o * CIN + c) * 9 + tap] = s;
    }
    if (i < kCh) {
        const float *db = part + (size_t)nch * N;
        float s = 0.f;
        for (int ch = 0; ch < nch; ch++) s += db[ch * kCh + i];
        gb[i] = s;
    }
}

// ---- head, backward ---------------------------------------------------------
constexpr int kF1 = kHid * P;                     // 23,104
constexpr int kF1PerThread = (kF1 + kThreads - 1) / kThreads;  // 91
constexpr int kHeadPart = kHeadParams + 1;        // + loss

__global__ __launch_bounds__(kThreads, 1) void sg_head_bwd(
    const __bf16 *__restrict__ h, const float *__restrict__ hp,
    const float *__restrict__ s_in, const float *__restrict__ f_in,
    const float *__restrict__ t_in, const float *__restrict__ y,
    __bf16 *__restrict__ e, float *__restrict__ part, int n, int bpc) {
    __shared__ float s[P];
    __shared__ float ds[P];
    __shared__ float df[kHid];
    __shared__ float red[kThreads];
    const int chunk = blockIdx.x, tid = threadIdx.x;
    const float *wh = hp, *F1 = hp + kCh + 1;
    const float *F2 = F1 + kF1 + kHid;
    const float inv_n = 1.f / (float)n;
    const int b0 = chunk * bpc;
    const int b1 = b0 + bpc < n ? b0 + bpc : n;

    float aF1[kF1PerThread];
#pragma unroll
    for (int k = 0; k < kF1PerThread; k++) aF1[k] = 0.f;
    float aF2 = 0.f, ac1 = 0.f, ac2 = 0.f, aloss = 0.f, awh = 0.f, abh = 0.f;
    const int c = tid & 63, g = tid >> 6;
    const float whc = wh[c];

    for (int b = b0; b < b1; b++) {
        const float t = t_in[b];
        const float ystar = 2.f * y[b] - 1.f;
        const float dz = 2.f * (t - ystar) * inv_n * (1.f - t * t);
        if (tid == 0) {
            aloss += (t - ystar) * (t - ystar);
            ac2 += dz;
        }
        if (tid < kHid) {
            const float fj = f_in[(size_t)b * kHid + tid];
            const float d = dz * F2[tid] * elu_grad(fj);
            df[tid] = d;
            aF2 += dz * fj;
            ac1 += d;
        }
        for (int p = tid; p < P; p += kThreads) s[p] = s_in[(size_t)b * P + p];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kF1PerThread; k++) {
            const int i = tid + k * kThreads;
            if (i < kF1) aF1[k] += df[i / P] * s[i % P];
        }
        for (int p = tid; p < P; p += kThreads) {
            float d = 0.f;
            for (int j = 0; j < kHid; j++) d += F1[j * P + p] * df[j];
            ds[p] = d * elu_grad(s[p]);
        }
        __syncthreads();
        for (int p = g; p < P; p += 4) {
            const size_t at = ((size_t)b * P + p) * kCh + c;
            const float hv = (float)h[at];
            const float d = ds[p];
            awh += d * hv;
            if (c == 0) abh += d;
            e[at] = (__bf16)(d * whc * elu_grad(hv));
        }
        __syncthreads();
    }
    float *dst = part + (size_t)chunk * kHeadPart;
    // wh and bh: sum the four pixel groups.
    red[tid] = awh;
    __syncthreads();
    if (tid < kCh) dst[tid] = red[tid] + red[tid + 64] + red[tid + 128] + red[tid + 192];
    __syncthreads();
    red[tid] = abh;
    __syncthreads();
    if (tid == 0) dst[kCh] = red[0] + red[64] + red[128] + red[192];
#pragma unroll
    for (int k = 0; k < kF1PerThread; k++) {
        const int i = tid + k * kThreads;
        if (i < kF1) dst[kCh + 1 + i] = aF1[k];
    }
    if (tid < kHid) {
        dst[kCh + 1 + kF1 + tid] = ac1;
        dst[kCh + 1 + kF1 + kHid + tid] = aF2;
    }
    if (tid == 0) {
        dst[kHeadParams - 1] = ac2;
        dst[kHeadParams] = aloss;
    }
}

__global__ __launch_bounds__(kThreads) void sg_head_reduce(
    const float *__restrict__ part, int nch, float inv_n,
    float *__restrict__ ghp, float *__restrict__ loss) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= kHeadPart) return;
    float s = 0.f;
    for (int ch = 0; ch < nch; ch++) s += part[(size_t)ch * kHeadPart + i];
    if (i < kHeadParams)
        ghp[i] = s;
    else
        *loss = s * inv_n;
}

__global__ __launch_bounds__(kThreads) void sg_adam(
    float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
    float *__restrict__ v, int count, float lr, float b1, float b2, float eps,
    float c1, float c2) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= count) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

int blocks(long long count) { return (int)((count + kThreads - 1) / kThreads); }

}  // namespace

hipError_t pack(const PackArgs &a, hipStream_t stream) {
    sg_pack<<<kPack0 + 2 * (kNConv - 1) * kPackL, kThreads, 0, stream>>>(a);
    return hipGetLastError();
}

hipError_t forward(const uint8_t *planes, const FwdArgs &a, uint16_t *act,
                   size_t map_elems, const float *hp, float *s, float *f,
                   float *t, float *win, int n, bool train,
                   hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    // One board per CU or fewer: eight waves on each.
    const int wm = n <= kWideBoards ? 2 : 1;
    const auto fn = wm == 2 ? (train ? sg_fwd<2, false> : sg_fwd<2, true>)
                            : (train ? sg_fwd<1, false> : sg_fwd<1, true>);
    fn<<<n, wm * kThreads, 0, stream>>>(planes, a, act, map_elems, hp, s, f, t,
                                        win);
    return hipGetLastError();
}

hipError_t conv_bwd(const uint16_t *e, const uint16_t *wpk,
                    const uint16_t *res, const uint16_t *mask, uint16_t *out,
                    int n, hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    sg_conv<<<n, kThreads, 0, stream>>>(
        (const __bf16 *)e, (const bf16x8 *)wpk, (const __bf16 *)res,
        (const __bf16 *)mask, (__bf16 *)out);
    return hipGetLastError();
}

size_t wgrad_part_floats(int cin, int n) {
    const int nch = chunks_for(n);
    return (size_t)nch * 9 * kCh * cin + (size_t)nch * kCh;
}

hipError_t wgrad(const void *in, int cin, const uint16_t *e, float *part,
                 float *gW, float *gb, int n, hipStream_t stream) {
    if (n <= 0) return hipErrorInvalidValue;
    const int nch = chunks_for(n);
    const int bpc = (n + nch - 1) / nch;
    const int used = (n + bpc - 1) / bpc;   // chunks that own boards
    const __bf16 *ev = (const __bf16 *)e;
    if (cin == 32) {
        sg_wgrad<32><<<9 * used, kThreads, 0, stream>>>(in, ev, part, n, bpc);
        sg_wgrad_reduce<32><<<blocks(9 * kCh * 32), kThreads, 0, stream>>>(
            part, used, gW, gb);
    } else if (cin == kCh) {
        sg_wgrad<kCh><<<9 * used, kThreads, 0, stream>>>(in, ev, part, n, bpc);
        sg_wgrad_reduce<kCh><<<blocks(9 * kCh * kCh), kThreads, 0, stream>>>(
            part, used, gW, gb);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

size_t head_part_floats(int n) { return (size_t)chunks_for(n) * kHeadPart; }

hipError_t head_bwd(const uint16_t *h, const float *hp, const float *s,
                    const float *f, const float *t, const float *y,
                    uint16_t *e, float *part, float *ghp, float *loss, int n,
                    hipStream_t stream) {
    if (n <= 0) return hipErrorInvalidValue;
    const int nch = chunks_for(n);
    const int bpc = (n + nch - 1) / nch;
    const int used = (n + bpc - 1) / bpc;
    sg_head_bwd<<<used, kThreads, 0, stream>>>((const __bf16 *)h, hp, s, f, t,
                                               y, (__bf16 *)e, part, n, bpc);
    sg_head_reduce<<<blocks(kHeadPart), kThreads, 0, stream>>>(
        part, used, 1.f / (float)n, ghp, loss);
    return hipGetLastError();
}

hipError_t adam(float *p, const float *g, float *m, float *v, int count,
                float lr, float beta1, float beta2, float eps, float c1,
                float c2, hipStream_t stream) {
    if (count <= 0) return hipSuccess;
    sg_adam<<<blocks(count), kThreads, 0, stream>>>(p, g, m, v, count, lr,
                                                    beta1, beta2, eps, c1, c2);
    return hipGetLastError();
}

}  // namespace sg
}  // namespace lz
