// lz_surrogate.h — device kernels of the learned playout surrogate (not part
// of the C ABI). The network:
//
//   a0 = elu(conv3x3(planes) + b0)                       32 -> 64
//   block k = 1..6: u = elu(conv(h) + b), h' = elu(conv(u) + b + h)
//   s  = elu(wh . h6 + bh)    (1x1, 64 -> 1)
//   f  = elu(F1 s + c1)       (361 -> 64)
//   t  = tanh(F2 . f + c2),   win rate (1 + t) / 2
//
// Activations and conv gradients live in HBM as BF16 HWC maps [n][361][64];
// parameters, gradients and Adam moments are FP32 (flat vector: per conv
// W[64][cin][3][3] then b[64]; then wh[64], bh, F1[64][361], c1[64], F2[64],
// c2). Convs run on MFMA with BF16 operands and FP32 accumulation.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lz {
namespace sg {

constexpr int kSide = 19;
constexpr int kP = kSide * kSide;
constexpr int kCh = 64;
constexpr int kNConv = 13;
constexpr int kHid = 64;
// Head parameters in flat order: wh[64], bh, F1[64][361], c1[64], F2[64], c2.
constexpr int kHeadParams = kCh + 1 + kHid * kP + kHid + kHid + 1;

inline int conv_cin(int layer) { return layer == 0 ? 32 : kCh; }
inline int conv_weights(int layer) { return kCh * conv_cin(layer) * 9; }

// Packed MFMA A-operand weights (BF16, 9 * cin * 64 values a conv) of every
// conv from its FP32 weights w: forward (wf) and, from conv 1 on,
// backward-data (wb: transposed, taps flipped).
struct PackArgs {
    const float *w[kNConv];
    uint16_t *wf[kNConv], *wb[kNConv];
};
hipError_t pack(const PackArgs &a, hipStream_t stream);

// The network's forward pass over n boards (planes u8 [n][32][361]): conv
// l's output to act + l * map_elems (BF16 [n][361][64]), the head's s
// [n][361], f [n][64] and t [n] (the backward pass reads them), win [n] =
// (1 + t) / 2 (may be null). w: packed forward weights, b: biases, hp: the
// head parameters. train: a backward pass follows and reads the maps.
struct FwdArgs {
    const uint16_t *w[kNConv];
    const float *b[kNConv];
};
hipError_t forward(const uint8_t *planes, const FwdArgs &a, uint16_t *act,
                   size_t map_elems, const float *hp, float *s, float *f,
                   float *t, float *win, int n, bool train,
                   hipStream_t stream);

// The backward pass to every pre-activation, for boards b0 .. b0 + n - 1 of
// a batch of `total` (loss mean_n (t - (2y - 1))^2) after forward(): the
// gradient at conv l's pre-activation into e + l * e_elems (BF16
// [n][361][64], board b0 first), and each board's kHeadRow floats of head
// gradients into hpart (indexed by board, as act, s, f, t and y are). w:
// packed backward-data weights (from conv 1 on).
constexpr int kHeadRow = 196;
struct BwdArgs {
    const uint16_t *w[kNConv];
};
hipError_t backward(const BwdArgs &a, const uint16_t *act, size_t map_elems,
                    const float *hp, const float *s, const float *f,
                    const float *t, const float *y, uint16_t *e,
                    size_t e_elems, float *hpart, int b0, int n, int total,
                    hipStream_t stream);

// Weight and bias gradients of every conv from n boards: e[l] its gradient
// maps, in[l] its input (u8 planes for conv 0). Written to w[l] (OIHW) and
// b[l], or added when `add`. With total > 0 (the last boards of a batch of
// `total`) also the head's gradients into ghp and the mean loss into *loss
// (device), from hpart and s. part must hold part_floats(n) floats.
struct WgradArgs {
    const void *in[kNConv];
    const uint16_t *e[kNConv];
    const void *zeros;  // 16 zero bytes
};
struct GradArgs {
    float *w[kNConv], *b[kNConv];
};
size_t part_floats(int n);
hipError_t wgrad(const WgradArgs &a, float *part, int n, const GradArgs &ga,
                 bool add, const float *hpart, const float *s, int total,
                 float *ghp, float *loss, hipStream_t stream);

// Adam (Kingma & Ba 2015, Algorithm 1) over count parameters; c1 = 1 -
// beta1^step, c2 = 1 - beta2^step.
hipError_t adam(float *p, const float *g, float *m, float *v, int count,
                float lr, float beta1, float beta2, float eps, float c1,
                float c2, hipStream_t stream);

}  // namespace sg
}  // namespace lz
