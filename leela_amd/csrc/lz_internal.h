// lz_internal.h — shared declarations of the HIP backend (not part of the
// C ABI). Kernels are compiled for gfx950 only.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lz {

// Largest board side the kernels accept (the reference nets are 19x19 only,
// Network.cpp:541-543,591-594,627-629).
constexpr int kMaxSide = 19;

// ---- FP32 plain form (conv_fp32.hip) --------------------------------------
// Its convs run on BF16 MFMA with every FP32 value split into three BF16
// parts. Input channels come in chunks of 32; activations between convs are
// [n][361][f32_stride(C)], the channels past C zero.
constexpr int f32_chunks(int cin) { return (cin + 31) / 32; }
constexpr int f32_stride(int c) { return f32_chunks(c) * 32; }

// Input planes per board the first conv may take (the reference's nets
// take 32) and the widest trunk conv of the FP32 form.
constexpr int kMaxInputPlanes = 64;
constexpr int kMaxTrunkChannels = 512;

// Conv activations (LZ_ACT_*).
constexpr int kActElu = 0, kActRelu = 1, kActNone = 2;

// What the FP32 conv epilogue applies after the bias: the activation, then
// (if bn_mean is set) bn_inv_std[o] * (v - bn_mean[o]).
struct ConvEpilogue {
    int act = kActElu;
    const float *bn_mean = nullptr;
    const float *bn_inv_std = nullptr;
};

// A conv's weights: `parts`, the three BF16 parts of each weight over its
// output channel's `scale` (a power of two, so that the channel's largest
// weight is 1 .. 2 and the parts of the others hold all their bits down to
// 2^-103 of it), as MFMA fragments; `plain`, the FP32 weights themselves.
// Trunk convs: parts [chunk][tap][part][m-tile][lane][8], plain
// [chunk][tap][m-tile][lane][8], scale [f32_stride(cout)]. The 3x3 head
// conv: parts [chunk][part][lane][8], plain [cin][9], scale [1].
struct SplitWeights {
    const uint16_t *parts;
    const float *scale, *plain;
};

// One same-padded conv over n 19x19 boards. in: byte planes [n][cin][361]
// (u8_input) or activations.
hipError_t conv_f32(int filter, bool u8_input, const void *in,
                    const SplitWeights &w, const float *bias, float *out,
                    int n, int cin, int cout, const ConvEpilogue &epi,
                    hipStream_t stream);

// Last 1-channel 3x3 conv + activation + softmax(T): raw/out [n][361].
hipError_t policy_head_f32(const float *in, const SplitWeights &w,
                           const float *b, float *raw, float *out, int n,
                           int cin, float temperature, int act,
                           hipStream_t stream);

// Last 1-channel conv + activation of the value net into h0 [n][361].
hipError_t value_headconv_f32(const float *in, const SplitWeights &w,
                              const float *b, float *h0, int n, int cin,
                              int act, hipStream_t stream);

// Value inner-product head over a batch: FC (P -> hidden) + ELU, FC
// (hidden -> 1), (1 + tanh) / 2. fc1_wt is the first FC transposed:
// [P][hidden]. Shared by every precision (the FCs stay FP32). n_dev (if not
// null) is a device-side board count that caps n when the kernel runs (a
// graph captured for n boards replayed on fewer).
hipError_t value_fc_head(const float *h0, const float *fc1_wt,
                         const float *fc1_b, const float *fc2_w,
                         const float *fc2_b, float *raw, float *out, int n,
                         int P, int hidden, hipStream_t stream,
                         const int *n_dev = nullptr);

}  // namespace lz
