// lz_conv_tile.h — implicit-GEMM convolution of an activation tile in LDS on
// 16-bit MFMA, shared by the persistent net kernels (fused_net.hip) and the
// surrogate's (surrogate.hip).
//
// A tile is HWC with zero halos; the waves of a workgroup form a grid over
// output channels x pixels, four of them along the pixels, six 16-pixel
// column tiles each (4 x 6 x 16 = 384 >= 361 pixels). Weights come from
// global memory packed in MFMA fragment order, [k-step][m-tile][lane][8],
// k-steps tap-major with 32 input channels each.
#pragma once

#include <hip/hip_runtime.h>

namespace lz {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename T>
struct Op;
template <>
struct Op<__bf16> {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    typedef __bf16 v4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ f32x4 mfma(v8 a, v8 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};
template <>
struct Op<_Float16> {
    typedef _Float16 v8 __attribute__((ext_vector_type(8)));
    typedef _Float16 v4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ f32x4 mfma(v8 a, v8 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};

constexpr int kWN = 4;                // waves along pixels
constexpr int kNT = 6;                // 16-pixel tiles per wave

// LDS bank layout of the tiles. A 16-byte ds_read (the B fragments of the
// convs) is served per half-wavefront, from 128 4-byte banks: the 32 lanes
// of a half-wave are conflict-free when their 16-byte units are distinct mod
// 32 (fitted to rocprofv3's SQ_LDS_BANK_CONFLICT over a set of lane
// patterns on gfx950). Lanes 0-31 of a fragment read 16 pixels x two
// 16-byte channel groups (units u*pixel + 0 and + 1, u = PS / 8). With u = 2
// mod 4 (PS = C + 16: 18 units for 128 channels, 10 for 64; 6 for the
// 32-plane input at 48) 16 consecutive pixels take the 16 even residues and
// the second channel group the odd ones. A 16-pixel column tile also wraps
// from the end of a board row to the next row, skipping the `halo` zero
// columns; the pad at the end of each row makes the row pitch, in units,
// congruent mod 32 to u times the S pixels of the row, so the pixels after
// a wrap continue the same residue sequence. row_pad is that pad, in
// elements (u * halo + pad = 0 mod 32 units).
constexpr int row_pad(int ps, int halo) {
    return 8 * ((((-halo * (ps / 8)) % 32) + 32) % 32);
}

// ELU of a trunk output that is about to be rounded to a 16-bit operand:
// exp(v) = 2^(v log2 e) on the hardware base-2 exponential (1 ulp), so
// exp(v) - 1 carries the same ~1e-7 absolute error as with the library
// expf, far below the 16-bit rounding that follows, without expf's
// range reduction, which dominated the epilogue's VALU time.
__device__ __forceinline__ float elu_operand(float v) {
    return v > 0.0f ? v
                    : __builtin_amdgcn_exp2f(v * 1.44269504088896341f) - 1.0f;
}

// One same-padded conv of the tile `act` (row pitch rp elements, pixel
// stride PS, CIN input channels) into acc[MTW][NT]: m-tiles mt0..mt0+MTW-1 (of MT in the
// packed weights) for the wave's column tiles; pb[t] is the lane's window
// origin in column tile t.
template <typename T, int F, int CIN, int MT, int MTW, int PS,
          int NT = kNT>
__device__ __forceinline__ void conv_tile(const T *act,
                                          const typename Op<T>::v8 *__restrict__ wpk,
                                          f32x4 (&acc)[MTW][NT],
                                          const int (&pb)[NT], int rp,
                                          int mt0, int lane,
                                          const float *__restrict__ bias =
                                              nullptr) {
    typedef typename Op<T>::v8 v8;
    constexpr int CB = CIN / 32;
    constexpr int STEPS = F * F * CB;
    const int g8 = (lane >> 4) * 8;
    // The accumulators start at the bias (when given): the epilogue then
    // has one add less per output.
#pragma unroll
    for (int m = 0; m < MTW; m++) {
        f32x4 init = {0.f, 0.f, 0.f, 0.f};
        if (bias) {
            const int o0 = (mt0 + m) * 16 + (lane >> 4) * 4;
#pragma unroll
            for (int r = 0; r < 4; r++) init[r] = bias[o0 + r];
        }
#pragma unroll
        for (int t = 0; t < NT; t++) acc[m][t] = init;
    }

    // (The empty asm keeps the compiler from hoisting the per-step
    // fragment addresses of a fully unrolled conv, the 1-channel head's,
    // out of the slot loop, where they would stay live, and spill, for the
    // whole kernel.)
    int lanev = lane;
    asm volatile("" : "+v"(lanev));
    const v8 *wl = wpk + mt0 * 64 + lanev;
    // Operands of k-step s, clamped to the last step (the loads issued past
    // the end re-read it and go unused).
    auto b_off = [&](int s) {
        s = s < STEPS ? s : STEPS - 1;
        const int tap = s / CB, cb = s % CB;
        return (tap / F) * rp + (tap % F) * PS + cb * 32 + g8;
    };
    auto a_at = [&](int s, int m) {
        s = s < STEPS ? s : STEPS - 1;
        return wl[(s * MT + m) * 64];
    };
    // B fragments (LDS) are loaded one k-step ahead into the other of two
    // register sets; the step loop is unrolled by two so that the sets
    // alternate without copies.
    v8 a[MTW], b0[NT], b1[NT];
#pragma unroll
    for (int m = 0; m < MTW; m++) a[m] = a_at(0, m);
#pragma unroll
    for (int t = 0; t < NT; t++)
        b0[t] = *reinterpret_cast<const v8 *>(act + pb[t] + g8);

    // Step s: acc += a * b while the B fragments of step s + 1 load into
    // bn. The MFMAs run m-tile by m-tile at raised wave priority; each A
    // fragment reloads with step s + 1's right after its last MFMA (a full
    // step of MFMAs ahead of its next use: the loads come from L2), and
    // the NT LDS reads are spread over the first half of the MFMAs.
    auto step = [&](const v8(&b)[NT], v8(&bn)[NT], int s) {
        const int off = b_off(s + 1);
#pragma unroll
        for (int t = 0; t < NT; t++)
            bn[t] = *reinterpret_cast<const v8 *>(act + pb[t] + off);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int m = 0; m < MTW; m++) {
#pragma unroll
            for (int t = 0; t < NT; t++)
                acc[m][t] = Op<T>::mfma(a[m], b[t], acc[m][t]);
            a[m] = a_at(s + 1, m);
        }
        constexpr int kMfma = MTW * NT;
        constexpr int kDsEvery = (kMfma / 2) / NT > 0 ? (kMfma / 2) / NT : 1;
        int ds = 0;
#pragma unroll
        for (int m = 0; m < MTW; m++) {
#pragma unroll
            for (int t = 0; t < NT; t++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
                if ((m * NT + t) % kDsEvery == kDsEvery - 1 && ds < NT) {
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // DS read
                    ds++;
                }
            }
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // VMEM read
        }
        __builtin_amdgcn_s_setprio(0);
    };
    for (int s = 0; s < STEPS; s += 2) {
        step(b0, b1, s);
        if (s + 1 < STEPS) step(b1, b0, s + 1);
    }
}

}  // namespace
}  // namespace lz
