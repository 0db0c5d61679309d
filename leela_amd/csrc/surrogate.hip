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
//   13 times, below one board per CU. At n = 4096: 1.61 ms (0.84 PFLOP/s),
//   against 3.37 ms for one launch per conv with its input staged from HBM
//   each time, with the same outputs to the bit: sums in the same order, the
//   library's expf. (The hardware base-2 exponential of a rounded product in
//   its place takes 0.28 ms less, but its absolute error is 6.9e-8 at most
//   against 4.5e-8.) Residuals read back from HBM instead of kept in
//   registers cost 0.7 ms of the 4096, stores of 8 bytes straight from the
//   accumulators 0.4 ms.
//
// Backward-data — sg_bwd
//   The same for the backward pass: one launch, a board's gradient map in
//   LDS from the head down to conv 0's output. dX = conv(dY; W') with
//   W'[c][o][tap] = W[o][c][8 - tap] (taps flipped), packed by sg_pack; the
//   epilogue adds the skip's gradient (kept in registers), multiplies by
//   ELU's derivative taken from the stored forward activation, and the map
//   goes to HBM for the weight gradients. n = 512: 242 us against 440 for
//   one launch per conv and 306 for the head's (the forward pass 215); 97 us
//   at n = 61. Besides the MFMAs it takes the mask map's trip through
//   registers after each conv.
//
// Weight gradients — sg_wgrad
//   dW[o][c][tap] = sum over boards and pixels of e[p][o] x[p + tap][c]: a
//   GEMM whose reduction runs over pixels. Both maps are staged as they lie
//   in HBM (pixel rows of 64 channels) and read with ds_read_b64_tr_b16,
//   which hands each lane four pixels of one channel: no transposed copies,
//   and a tap is only another pixel address, so one staging serves all nine.
//   All convs in one launch; a workgroup takes one conv and a run of boards,
//   half a board at a time, each of its eight waves 16 input channels x 9
//   taps x 64 output channels (144 accumulators) over half the pixels.
//   sg_reduce sums the partials in a fixed order (deterministic) into OIHW.
//   Bound at n = 512: 0.7 GB of maps read (134 us at this card's copy rate)
//   and 173 GFLOP; 213-229 us, of which the copies alone take 140 and the MFMAs
//   alone 137 (two buffers do not hide all of the one behind the other; a
//   k-step's copies issued between its MFMAs instead of ahead of them
//   measured 217). Nine transposed copies of each map, one per tap, took
//   3.8 ms.
//
// Head (ELU activations), loss, Adam: FP32 (the head is 0.2% of the FLOPs).
#include "lz_conv_tile.h"
#include "lz_surrogate.h"

namespace lz {
namespace sg {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

constexpr int S = kSide, P = kP;
constexpr int HS = S + 2, HP = HS * HS;   // halo frame 21 x 21
constexpr int kThreads = 256;
// Workgroups per conv of a weight-gradient launch, at most: 13 x 19 = 247,
// one on each CU.
constexpr int kMaxChunks = 19;
constexpr int kPart = 9 * kCh * kCh;  // floats of a weight-gradient partial
// Batches of at most this many boards (one per CU) use eight waves a board:
// 116 us at n = 1 and 121 at 256, against 155-158 with four; from 257 on
// a CU holds two boards and four waves each are faster (193 against 213 us
// at 257, 405 against 429 at 1024).
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
int boards_per_chunk(int n) { return (n + chunks_for(n) - 1) / chunks_for(n); }

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

// Epilogue of a forward conv: + bias, + residual, ELU, BF16 into the tile.
// acc's lane holds four consecutive channels of one pixel per fragment.
// bias: the conv's 64, in LDS. keep: the lane's outputs of the last even
// conv, which are the residual of an even conv (kRes) and are replaced by its
// outputs (kKeep). (The sums in this order and the library's expf: the
// outputs are to the bit those of one launch per conv.)
template <bool kRes, bool kKeep, int MTW>
__device__ __forceinline__ void sg_store_fwd(__bf16 *tile,
                                             const f32x4 (&acc)[MTW][kNT],
                                             bf16x4 (&keep)[MTW][kNT],
                                             const float *bias, int mt0,
                                             const int (&pb)[kNT],
                                             const int (&pix)[kNT], int lane) {
    const int g4 = (lane >> 4) * 4;
#pragma unroll
    for (int m = 0; m < MTW; m++) {
        const int o = (mt0 + m) * 16 + g4;
        const f32x4 bo = *(const f32x4 *)(bias + o);
#pragma unroll
        for (int t = 0; t < kNT; t++) {
            bf16x4 v;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float d = acc[m][t][r] + bo[r];
                v[r] = (__bf16)elu(kRes ? d + (float)keep[m][t][r] : d);
            }
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
    __shared__ __attribute__((aligned(16))) float s_bias[kNConv * kCh];
    const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int mt0 = (w / kWN) * MTW;
    const bf16x8 zero8 = {};
    __bf16 *maps = (__bf16 *)act + (size_t)b * P * kCh;

#pragma unroll
    for (int l = 0; l < kNConv; l++)
        if (tid < kCh) s_bias[l * kCh + tid] = a.b[l][tid];
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
            tile, (const bf16x8 *)a.w[0], acc, pbi, kInRP, mt0, lane);
        __syncthreads();
        for (int i = tid * 8; i < kTile; i += T * 8)
            *(bf16x8 *)(tile + i) = zero8;
        __syncthreads();
        sg_store_fwd<false, true, MTW>(tile, acc, keep, s_bias, mt0, pb, pix,
                                       lane);
        __syncthreads();
    }
    // The map of a conv's input goes out between its MFMAs and its epilogue:
    // loads and stores retire in order, so stores ahead of a conv would
    // hold up its weight loads, and here the epilogue's math covers them.
    for (int l = 1; l < kNConv; l += 2) {
        f32x4 acc[MTW][kNT];
        conv_tile<__bf16, 3, kCh, MT, MTW, kPS>(
            tile, (const bf16x8 *)a.w[l], acc, pb, kRP, mt0, lane);
        sg_copy_out<T, kStream>(tile, maps + (l - 1) * map_elems, tid);
        __syncthreads();
        sg_store_fwd<false, false, MTW>(tile, acc, keep, s_bias + l * kCh, mt0,
                                        pb, pix, lane);
        __syncthreads();
        conv_tile<__bf16, 3, kCh, MT, MTW, kPS>(
            tile, (const bf16x8 *)a.w[l + 1], acc, pb, kRP, mt0, lane);
        sg_copy_out<T, kStream>(tile, maps + l * map_elems, tid);
        __syncthreads();
        sg_store_fwd<true, true, MTW>(tile, acc, keep, s_bias + (l + 1) * kCh,
                                      mt0, pb, pix, lane);
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

// ---- the backward pass ----------------------------------------------------------
constexpr int kF1 = kHid * P;  // 23,104
// A board's share of the small head gradients, one row per board:
// wh[64], c1[64] (the gradient at f's pre-activation), F2[64], bh, c2, loss.
constexpr int kHpWh = 0, kHpC1 = kCh, kHpF2 = kCh + kHid;
constexpr int kHpBh = kCh + 2 * kHid, kHpC2 = kHpBh + 1, kHpLoss = kHpBh + 2;
static_assert(kHpLoss < kHeadRow && kHeadRow % 4 == 0, "head gradient row");

// Epilogue of a backward-data conv: (acc + skip) * ELU'(mask), BF16. The
// tile holds the mask map's board (copied there after the conv): each lane
// reads its four channels of a pixel and writes the result in their place.
// keep: the lane's values of the last even map, the skip of the next
// (kRes), replaced by the outputs (kKeep).
template <bool kRes, bool kKeep, int MTW>
__device__ __forceinline__ void sg_store_bwd(__bf16 *tile,
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
            bf16x4 *at = (bf16x4 *)(tile + pb[t] + kRP + kPS + o);
            const bf16x4 mv = *at;
            bf16x4 v;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float d =
                    kRes ? acc[m][t][r] + (float)keep[m][t][r] : acc[m][t][r];
                v[r] = (__bf16)(d * elu_grad((float)mv[r]));
            }
            if (kKeep) keep[m][t] = v;
            if (pix[t] >= 0) *at = v;
        }
    }
}

// Part `part` of a board's map from HBM into registers (load) and on into
// the tile (put), 16 bytes a lane: the whole map with 512 threads, half of it
// with 256 (six loads of registers beside the accumulators).
template <int T>
struct MapRegs {
    static constexpr int N = 6, kParts = 2 * kThreads / T;
    static_assert(N * kParts * T >= P * 8, "parts cover the map");
    bf16x8 v[N];
    __device__ __forceinline__ void load(const __bf16 *map, int part, int tid) {
#pragma unroll
        for (int k = 0; k < N; k++) {
            const int i = tid + (part * N + k) * T;
            if (i < P * 8) v[k] = *(const bf16x8 *)(map + i * 8);
        }
    }
    __device__ __forceinline__ void put(__bf16 *tile, int part, int tid) const {
#pragma unroll
        for (int k = 0; k < N; k++) {
            const int i = tid + (part * N + k) * T, p = i >> 3;
            if (i < P * 8)
                *(bf16x8 *)(tile + (p / S + 1) * kRP + (p % S + 1) * kPS +
                            (i & 7) * 8) = v[k];
        }
    }
};

// Board b0 + blockIdx.x. e: maps of this launch's boards (gradient at conv
// l's pre-activation at e + l * e_elems); act, s, f, t, y, hpart: by board.
// Wave grid as sg_fwd's.
template <int kWM>
__global__ __launch_bounds__(kWM * kThreads, 2) void sg_bwd(
    BwdArgs a, const uint16_t *__restrict__ act, size_t map_elems,
    const float *__restrict__ hp, const float *__restrict__ s_in,
    const float *__restrict__ f_in, const float *__restrict__ t_in,
    const float *__restrict__ y, uint16_t *__restrict__ e, size_t e_elems,
    float *__restrict__ hpart, int b0, float inv_n) {
    constexpr int T = kWM * kThreads, W = kWM * 4;
    constexpr int MT = kCh / 16, MTW = MT / kWM;
    __shared__ __attribute__((aligned(16))) __bf16 tile[kTile];
    __shared__ float s[P];
    __shared__ float ds[P];
    __shared__ float df[kHid];
    __shared__ float red[W][kCh];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int b = b0 + blockIdx.x;
    const int mt0 = (w / kWN) * MTW;
    const __bf16 *amaps = (const __bf16 *)act + (size_t)b * P * kCh;
    __bf16 *emaps = (__bf16 *)e + (size_t)blockIdx.x * P * kCh;
    float *row = hpart + (size_t)b * kHeadRow;

    // Head. hp: wh[64], bh, F1[64][361], c1[64], F2[64], c2.
    const float *F1 = hp + kCh + 1, *F2 = F1 + kF1 + kHid;
    const float t = t_in[b], ystar = 2.f * y[b] - 1.f;
    const float dz = 2.f * (t - ystar) * inv_n * (1.f - t * t);
    MapRegs<T> mask;
    constexpr int kParts = MapRegs<T>::kParts;
    const __bf16 *last = amaps + (kNConv - 1) * map_elems;
    mask.load(last, 0, tid);
    if (tid < kHid) {
        const float fj = f_in[(size_t)b * kHid + tid];
        const float d = dz * F2[tid] * elu_grad(fj);
        df[tid] = d;
        row[kHpC1 + tid] = d;
        row[kHpF2 + tid] = dz * fj;
    }
    if (tid == 0) {
        row[kHpC2] = dz;
        row[kHpLoss] = (t - ystar) * (t - ystar);
    }
    for (int p = tid; p < P; p += T) s[p] = s_in[(size_t)b * P + p];
    const bf16x8 zero8 = {};
    for (int i = tid * 8; i < kTile; i += T * 8)
        *(bf16x8 *)(tile + i) = zero8;
    __syncthreads();
    for (int p = tid; p < P; p += T) {
        float d = 0.f;
#pragma unroll 16
        for (int j = 0; j < kHid; j++) d += F1[j * P + p] * df[j];
        ds[p] = d * elu_grad(s[p]);
    }
    __syncthreads();
    // Map 12, and wh's gradient: a thread has 8 fixed channels.
    {
        const int c8 = tid & 7;
        float wh[8], dw[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            wh[k] = hp[c8 * 8 + k];
            dw[k] = 0.f;
        }
        for (int part = 0; part < kParts; part++) {
            if (part) mask.load(last, part, tid);
#pragma unroll
            for (int k = 0; k < MapRegs<T>::N; k++) {
                const int i = tid + (part * MapRegs<T>::N + k) * T;
                if (i >= P * 8) break;
                const float d = ds[i >> 3];
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    const float hv = (float)mask.v[k][q];
                    dw[q] += d * hv;
                    mask.v[k][q] = (__bf16)(d * wh[q] * elu_grad(hv));
                }
            }
            mask.put(tile, part, tid);
        }
#pragma unroll
        for (int q = 0; q < 8; q++) {
            for (int o = 8; o < 64; o <<= 1) dw[q] += __shfl_xor(dw[q], o, 64);
            if (lane < 8) red[w][c8 * 8 + q] = dw[q];
        }
    }
    __syncthreads();
    if (tid < kCh) {
        float v = 0.f;
#pragma unroll
        for (int i = 0; i < W; i++) v += red[i][tid];
        row[kHpWh + tid] = v;
    }
    if (w == W - 1) {
        float v = 0.f;
        for (int p = lane; p < P; p += 64) v += ds[p];
        v = wave_sum(v);
        if (lane == 0) row[kHpBh] = v;
    }

    int pb[kNT], pix[kNT];
    sg_geom(w % kWN, lane, pb, pix);
    bf16x4 keep[MTW][kNT];
#pragma unroll
    for (int m = 0; m < MTW; m++)
#pragma unroll
        for (int q = 0; q < kNT; q++)
            keep[m][q] = *(const bf16x4 *)(tile + pb[q] + kRP + kPS +
                                           (mt0 + m) * 16 + (lane >> 4) * 4);
    // Conv l turns map l (in the tile) into map l - 1. After its MFMAs the
    // map in the tile goes out and its ELU mask comes in.
    auto swap = [&](int l) {
        const __bf16 *m = amaps + (l - 1) * map_elems;
        mask.load(m, 0, tid);
        sg_copy_out<T, false>(tile, emaps + l * e_elems, tid);
        __syncthreads();
#pragma unroll
        for (int part = 0; part < kParts; part++) {
            if (part) mask.load(m, part, tid);
            mask.put(tile, part, tid);
        }
        __syncthreads();
    };
    for (int l = kNConv - 1; l >= 1; l -= 2) {
        f32x4 acc[MTW][kNT];
        conv_tile<__bf16, 3, kCh, MT, MTW, kPS>(
            tile, (const bf16x8 *)a.w[l], acc, pb, kRP, mt0, lane);
        swap(l);
        sg_store_bwd<false, false, MTW>(tile, acc, keep, mt0, pb, pix, lane);
        __syncthreads();
        conv_tile<__bf16, 3, kCh, MT, MTW, kPS>(
            tile, (const bf16x8 *)a.w[l - 1], acc, pb, kRP, mt0, lane);
        swap(l - 1);
        sg_store_bwd<true, true, MTW>(tile, acc, keep, mt0, pb, pix, lane);
        __syncthreads();
    }
    sg_copy_out<T, false>(tile, emaps, tid);
}

// ---- weight gradients -----------------------------------------------------------
// A stage is half a board: output rows y0 .. y0 + 9 (190 pixels) or + 8
// (171), reduced in six k-steps of 32 pixels, and the input's rows y0 - 1 ..
// y0 + 10 in a 12 x 24 frame; zeros past the half and off the board. Two
// buffers: the next stage's copies (direct global-to-LDS, whole pixels of
// 128 bytes, zeros read from a zero block) run under this stage's MFMAs.
// Within a pixel the four groups of 16 channels are permuted: group m lies
// at place m ^ (pixel / 2 % 4), so that a transposed read of 16 pixels in a
// row touches every bank the same number of times; the frame's width keeps
// the permutation from row to row, so a tap's row is a constant offset.
constexpr int kWgThreads = 512;
constexpr int kHalfRows = 10, kHalfPix = 192;
constexpr int kFW = 24, kFrameRows = 12, kFramePix = kFW * kFrameRows;
constexpr int kStage = kCh * (kHalfPix + kFramePix);  // elements
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

__device__ __forceinline__ int chan_place(int m, int pixel) {
    return (m ^ (pixel >> 1 & 3)) * 16;
}

// The transposed read: the 16 lanes of a group name four pixel rows (lane
// i row i / 4, channels 4 (i % 4) ..); lane i gets channel i of the four.
// The two reads of a fragment are 16 pixels apart (any order of the pixels
// does, the same for both operands).
__device__ __forceinline__ bf16x8 tr_frag(const __bf16 *lo, const __bf16 *hi) {
    union {
        s16x4 h[2];
        bf16x8 v;
    } u;
    u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)lo);
    u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)hi);
    return u.v;
}

// 16 bytes a lane from global memory to LDS at dst + 16 * lane (dst the same
// in the whole wave). Written in assembly because the compiler makes every
// LDS read after the builtin wait for the copy; the caller waits for all of
// them (vmcnt(0)) before the barrier that hands the buffer over. The
// instruction has no register output.
__device__ __forceinline__ void copy_async(const void *src, __bf16 *dst) {
    const uint32_t at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(
        __attribute__((address_space(3))) __bf16 *)dst);
    asm volatile(
        "s_mov_b32 m0, %0\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, off"
        :
        : "s"(at), "v"(src)
        : "memory", "m0");
}

// One conv over boards b .. b1. kPlanes: conv 0, whose 32 input planes
// (bytes) go to LDS through registers.
template <bool kPlanes>
__device__ __forceinline__ void wgrad_boards(const void *in, const __bf16 *e,
                                             const void *zeros, float *part,
                                             float *bpart, int b, int b1,
                                             __bf16 *buf) {
    constexpr int CIN = kPlanes ? 32 : kCh;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, i16 = lane & 15;
    const int cg = w & 3, ks0 = (w >> 2) * 3;  // 16 input channels, k-steps
    const bool mine = cg * 16 < CIN;
    f32x4 acc[9][4];
#pragma unroll
    for (int tap = 0; tap < 9; tap++)
#pragma unroll
        for (int m = 0; m < 4; m++) acc[tap][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    float db[2] = {0.f, 0.f};
    // The lane's pixel in read h of k-step k: 32 k + 16 h + j0.
    const int j0 = ks0 * 32 + g * 4 + (i16 >> 2), c4 = (i16 & 3) * 4;
    int eat[4], xat[3][2][3];
#pragma unroll
    for (int m = 0; m < 4; m++) eat[m] = j0 * kCh + chan_place(m, j0) + c4;
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            int j = j0 + k * 32 + h * 16;
            j = j < kHalfRows * S ? j : kHalfRows * S - 1;
#pragma unroll
            for (int dx = 0; dx < 3; dx++) {
                const int q = (j / S) * kFW + j % S + dx;
                xat[k][h][dx] =
                    (kHalfPix + q) * kCh + chan_place(cg, q) + c4;
            }
        }

    // Stage st of the run (two per board) into buffer `to`: copies of eight
    // pixels, 24 of e and 36 of the input. Conv 0: a thread takes 16 planes
    // of a point on the board; the frame's side columns stay zero.
    const uint8_t *pl = (const uint8_t *)in;
    uint8_t px[16];
    const int pq = tid % (kFrameRows * S), pc = tid / (kFrameRows * S);
    auto issue = [&](int st, __bf16 *to) {
        const int board = b + (st >> 1), y0 = st & 1 ? kHalfRows : 0;
        const int npx = st & 1 ? (S - kHalfRows) * S : kHalfRows * S;
        const __bf16 *es = e + ((size_t)board * P + y0 * S) * kCh;
        const __bf16 *xs =
            (const __bf16 *)in + ((size_t)board * P + (y0 - 1) * S) * kCh;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int u = k * 8 + w, p8 = lane >> 3;
            if (u < kHalfPix / 8) {
                const int j = u * 8 + p8;
                const int ch = ((lane & 7) ^ (j >> 1 & 3) << 1) * 8;
                copy_async(j < npx ? es + j * kCh + ch : zeros,
                           to + u * 8 * kCh);
            } else if (!kPlanes && u < (kHalfPix + kFramePix) / 8) {
                const int q = (u - kHalfPix / 8) * 8 + p8;
                const int ch = ((lane & 7) ^ (q >> 1 & 3) << 1) * 8;
                const int r = q / kFW, x = q % kFW - 1, yy = y0 - 1 + r;
                const bool on = x >= 0 && x < S && yy >= 0 && yy < S;
                copy_async(on ? xs + (r * S + x) * kCh + ch : zeros,
                           to + u * 8 * kCh);
            }
        }
        if (kPlanes && pc < 2) {
            const int yy = y0 - 1 + pq / S;
            const bool on = yy >= 0 && yy < S;
#pragma unroll
            for (int c = 0; c < 16; c++)
                px[c] = on ? pl[((size_t)board * 32 + pc * 16 + c) * P +
                                yy * S + pq % S]
                           : 0;
        }
    };
    auto settle = [&](__bf16 *to) {
        if (kPlanes && pc < 2) {
            bf16x8 v[2];
#pragma unroll
            for (int c = 0; c < 16; c++) v[c >> 3][c & 7] = (__bf16)(float)px[c];
            const int q = (pq / S) * kFW + pq % S + 1;
            __bf16 *at = to + (kHalfPix + q) * kCh + chan_place(pc, q);
            *(bf16x8 *)at = v[0];
            *(bf16x8 *)(at + 8) = v[1];
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };

    const int stages = 2 * (b1 - b);
    if (kPlanes) {
        const bf16x8 zero8 = {};
        for (int i = tid * 8; i < 2 * kStage; i += kWgThreads * 8)
            *(bf16x8 *)(buf + i) = zero8;
        __syncthreads();
    }
    issue(0, buf);
    settle(buf);
    for (int st = 0; st < stages; st++) {
        const __bf16 *cur = buf + (st & 1) * kStage;
        __bf16 *nxt = buf + (~st & 1) * kStage;
        if (st + 1 < stages) issue(st + 1, nxt);
        if (mine) {
#pragma unroll
            for (int k = 0; k < 3; k++) {
                // (A k-step's reads stay in it: all three's do not fit the
                // registers beside the accumulators.)
                __builtin_amdgcn_sched_barrier(0);
                bf16x8 af[4];
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    const __bf16 *at = cur + eat[m] + k * 32 * kCh;
                    af[m] = tr_frag(at, at + 16 * kCh);
                }
#pragma unroll
                for (int tap = 0; tap < 9; tap++) {
                    const __bf16 *at = cur + (tap / 3) * kFW * kCh;
                    const bf16x8 bv = tr_frag(at + xat[k][0][tap % 3],
                                              at + xat[k][1][tap % 3]);
#pragma unroll
                    for (int m = 0; m < 4; m++)
                        acc[tap][m] = mfma(af[m], bv, acc[tap][m]);
                }
#pragma unroll
                for (int m = 0; m < 4; m++)
                    if (m % (CIN / 16) == cg) {
#pragma unroll
                        for (int q = 0; q < 8; q++)
                            db[m / (CIN / 16)] += (float)af[m][q];
                    }
            }
        }
        if (st + 1 < stages) settle(nxt);
    }
    if (!mine) return;
    // Partials [k half][tap][o][c], bias sums [k half][o].
    float *dst = part + (w >> 2) * kPart + cg * 16 + i16;
#pragma unroll
    for (int tap = 0; tap < 9; tap++)
#pragma unroll
        for (int m = 0; m < 4; m++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                dst[(tap * kCh + m * 16 + g * 4 + r) * CIN] = acc[tap][m][r];
#pragma unroll
    for (int i = 0; i < kCh / CIN; i++) {
        db[i] += __shfl_xor(db[i], 16, 64);
        db[i] += __shfl_xor(db[i], 32, 64);
        if (lane < 16)
            bpart[(w >> 2) * kCh + (i * (CIN / 16) + cg) * 16 + lane] = db[i];
    }
}

// Workgroup (conv l, chunk of bpc boards) = blockIdx / chunks, % chunks.
// part: [l][chunk][k half][kPart], then bias sums [l][chunk][k half][64].
__global__ __launch_bounds__(kWgThreads, 2) void sg_wgrad(
    WgradArgs a, float *__restrict__ part, int n, int bpc, int chunks) {
    __shared__ __attribute__((aligned(1024))) __bf16 buf[2 * kStage];
    const int l = blockIdx.x / chunks, chunk = blockIdx.x % chunks;
    const int b0 = chunk * bpc, b1 = b0 + bpc < n ? b0 + bpc : n;
    float *p = part + (size_t)blockIdx.x * 2 * kPart;
    float *bp = part + (size_t)kNConv * chunks * 2 * kPart +
                (size_t)blockIdx.x * 2 * kCh;
    const __bf16 *e = (const __bf16 *)a.e[l];
    if (l == 0)
        wgrad_boards<true>(a.in[0], e, a.zeros, p, bp, b0, b1, buf);
    else
        wgrad_boards<false>(a.in[l], e, a.zeros, p, bp, b0, b1, buf);
}

// ---- sums of partials -------------------------------------------------------------
// Every sum of a backward pass in one launch, by blocks: conv 0's weights,
// the other convs', all biases, and (with the last boards) F1's gradient
// sum_b df[b][j] s[b][p] and the rows of small head gradients. A block
// splits each sum over slices of threads (one load after another would be
// one memory latency per partial) and adds the slices in order.
constexpr int kRedThreads = 1024;
constexpr int kRed0 = 9 * kCh * 32 / 4 / 64, kRedL = kPart / 4 / 64;
constexpr int kRedBias = kRed0 + (kNConv - 1) * kRedL;
constexpr int kRedF1 = kRedBias + 1;
constexpr int kF1PB = (P + 63) / 64;
constexpr int kRedSmall = kRedF1 + kF1PB * (kHid / 4);
constexpr int kRedBlocks = kRedSmall + (kHpLoss + 1 + 31) / 32;

__global__ __launch_bounds__(kRedThreads) void sg_reduce(
    const float *__restrict__ part, int chunks, GradArgs ga, bool add,
    const float *__restrict__ hpart, const float *__restrict__ s, int n,
    float inv_n, float *__restrict__ ghp, float *__restrict__ loss) {
    __shared__ f32x4 red[16][64];
    const int tid = threadIdx.x, q = tid & 63, sl = tid >> 6;
    const int blk = blockIdx.x;
    if (blk < kRedBias) {
        const int l = blk < kRed0 ? 0 : 1 + (blk - kRed0) / kRedL;
        const int cin = l ? kCh : 32;
        const int at = ((l ? (blk - kRed0) % kRedL : blk) * 64 + q) * 4;
        const float *src = part + (size_t)l * chunks * 2 * kPart + at;
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
        for (int c = sl; c < 2 * chunks; c += 16)
            v += *(const f32x4 *)(src + (size_t)c * kPart);
        red[sl][q] = v;
        __syncthreads();
        if (sl) return;
        for (int i = 1; i < 16; i++) v += red[i][q];
        const int tap = at / (kCh * cin), o = (at / cin) % kCh, c = at % cin;
        float *g = ga.w[l] + (o * cin + c) * 9 + tap;
        for (int r = 0; r < 4; r++) g[r * 9] = add ? g[r * 9] + v[r] : v[r];
    } else if (blk < kRedF1) {
        if (tid >= kNConv * kCh) return;
        const int l = tid / kCh, o = tid % kCh;
        const float *src = part + (size_t)kNConv * chunks * 2 * kPart +
                           (size_t)l * chunks * 2 * kCh + o;
        float v = add ? ga.b[l][o] : 0.f;
#pragma unroll 8
        for (int c = 0; c < 2 * chunks; c++) v += src[c * kCh];
        ga.b[l][o] = v;
    } else if (blk < kRedSmall) {
        const int j0 = (blk - kRedF1) / kF1PB * 4;
        const int p = (blk - kRedF1) % kF1PB * 64 + q;
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        if (p < P) {
#pragma unroll 8
            for (int b = sl; b < n; b += 16)
                v += *(const f32x4 *)(hpart + (size_t)b * kHeadRow + kHpC1 + j0) *
                     s[(size_t)b * P + p];
        }
        red[sl][q] = v;
        __syncthreads();
        if (sl || p >= P) return;
        for (int i = 1; i < 16; i++) v += red[i][q];
        for (int j = 0; j < 4; j++) ghp[kCh + 1 + (j0 + j) * P + p] = v[j];
    } else {
        float *r1 = (float *)red;  // [32][33]
        const int o = (blk - kRedSmall) * 32 + (tid & 31), s32 = tid >> 5;
        float v = 0.f;
        if (o <= kHpLoss) {
#pragma unroll 8
            for (int b = s32; b < n; b += 32) v += hpart[(size_t)b * kHeadRow + o];
        }
        r1[s32 * 33 + (tid & 31)] = v;
        __syncthreads();
        if (s32 || o > kHpLoss) return;
        for (int i = 1; i < 32; i++) v += r1[i * 33 + tid];
        if (o < kHpC1)
            ghp[o] = v;
        else if (o < kHpF2)
            ghp[kCh + 1 + kF1 + o - kHpC1] = v;
        else if (o < kHpBh)
            ghp[kCh + 1 + kF1 + kHid + o - kHpF2] = v;
        else if (o == kHpBh)
            ghp[kCh] = v;
        else if (o == kHpC2)
            ghp[kHeadParams - 1] = v;
        else
            *loss = v * inv_n;
    }
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

size_t part_floats(int n) {
    return (size_t)kNConv * chunks_for(n) * 2 * (kPart + kCh);
}

hipError_t backward(const BwdArgs &a, const uint16_t *act, size_t map_elems,
                    const float *hp, const float *s, const float *f,
                    const float *t, const float *y, uint16_t *e,
                    size_t e_elems, float *hpart, int b0, int n, int total,
                    hipStream_t stream) {
    if (n <= 0) return hipErrorInvalidValue;
    const int wm = n <= kWideBoards ? 2 : 1;
    const auto fn = wm == 2 ? sg_bwd<2> : sg_bwd<1>;
    fn<<<n, wm * kThreads, 0, stream>>>(a, act, map_elems, hp, s, f, t, y, e,
                                        e_elems, hpart, b0, 1.f / (float)total);
    return hipGetLastError();
}

hipError_t wgrad(const WgradArgs &a, float *part, int n, const GradArgs &ga,
                 bool add, const float *hpart, const float *s, int total,
                 float *ghp, float *loss, hipStream_t stream) {
    if (n <= 0) return hipErrorInvalidValue;
    const int bpc = boards_per_chunk(n);
    const int used = (n + bpc - 1) / bpc;  // chunks that own boards
    sg_wgrad<<<kNConv * used, kWgThreads, 0, stream>>>(a, part, n, bpc, used);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    sg_reduce<<<total > 0 ? kRedBlocks : kRedF1, kRedThreads, 0, stream>>>(
        part, used, ga, add, hpart, s, total,
        total > 0 ? 1.f / (float)total : 0.f, ghp, loss);
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
