// mc_playout.hip — the reference's pattern playout policy on the GPU: one
// playout per wavefront, running the same source as the host (mc_core.h), so
// each playout is the same move sequence and final score as the host's for
// the same position and seed (Playout::run / mc_owner, Playout.cpp:51-113,
// 174-217, with FastState::play_random_move, FastState.cpp:168-255).
//
// The policy's state is pointer-chasing over a FastBoard-like board (string
// lists, the empty list, the candidate list): a playout is one long chain of
// dependent reads, so their latency is its time. The board and the first
// candidates live in LDS (7.3 KB a playout, 20 wavefronts a CU); every lane
// runs the serial steps alike, and the lanes share what is independent: the
// scan of the empty list for a playable point, and the scoring of the
// candidates. Wavefronts draw playouts from a counter until none is left.
// Bound: the instructions of the serial steps (20 wavefronts a CU or 8 run
// at the same rate). 19x19, 16,384 playouts 23.6 ms (694k/s), 65,536 77 ms
// (847k/s), 256 7.0 ms; with one playout per lane and the state in global
// memory 152, 244 and 141 ms.
// This file is compiled with -ffp-contract=off: the scores' products and
// running sums must round exactly as the host's do.
#include <hip/hip_runtime.h>

#include "lz_encoder.h"
#include "mc_core.h"

namespace lz {
namespace {

// Candidates beside the board, and the rest of a list in global memory
// (rarely reached: a move generation holds a few dozen).
constexpr int kFastMoves = 64;
constexpr int kSpillMoves = mc::kDevMoves - kFastMoves;

struct WaveMoves {
    int n;
    bool overflow;
    mc::Move *rest;
    mc::Move first[kFastMoves];
    __device__ void clear() {
        n = 0;
        overflow = false;
    }
    __device__ bool empty() const { return n == 0; }
    __device__ int size() const { return n; }
    __device__ mc::Move get(int i) const {
        if (i < kFastMoves) return first[i];
        return rest[i - kFastMoves];
    }
    __device__ void set(int i, const mc::Move &x) {
        if (i < kFastMoves)
            first[i] = x;
        else
            rest[i - kFastMoves] = x;
    }
    __device__ void add_back(int flag, const mc::TablesView &t) {
        mc::Move x = get(n - 1);
        x.add(flag, t);
        set(n - 1, x);
    }
    __device__ void push(int v, int flag, const mc::TablesView &t) {
        if (n >= mc::kDevMoves) {
            overflow = true;
            return;
        }
        mc::Move x;
        x.word = (uint32_t)(v + 1) << 22;
        x.score = 1.0f;
        x.add(flag, t);
        set(n++, x);
    }
};

// The lanes of the workgroup's one wavefront share the steps.
struct WaveExec {
    template <class F>
    __device__ static int first(int n, F f) {
        for (int base = 0; base < n; base += 64) {
            const int i = base + (int)threadIdx.x;
            const bool hit = i < n && f(i);
            const uint64_t b = __builtin_amdgcn_ballot_w64(hit);
            if (b) return base + __builtin_ctzll(b);
        }
        return -1;
    }
    template <class F>
    __device__ static void each(int n, F f) {
        __syncthreads();
        for (int i = (int)threadIdx.x; i < n; i += 64) f(i);
        __syncthreads();
    }
};

using WaveState = mc::PlayStateT<WaveMoves, WaveExec>;

__global__ __launch_bounds__(64) void pat_zero(uint32_t *half_wins,
                                               uint32_t *overflow, int npos,
                                               unsigned long long *next) {
    const int i = blockIdx.x * 64 + threadIdx.x;
    if (i == 0) *next = 0;
    if (i < npos) {
        half_wins[i] = 0;
        overflow[i] = 0;
    }
}

// The npos x nplay grid of playouts; playout j of position p is seeded
// playout_seed(seed0 + p, j) with two outputs discarded. Outcomes are summed
// as half points per position.
__global__ __launch_bounds__(64, 5) void pat_playout_kernel(
    const EncRecord *__restrict__ recs, int npos, int nplay, uint32_t seed0,
    mc::TablesView tables, mc::Move *spill, unsigned long long *next,
    uint32_t *half_wins, uint32_t *overflow) {
    __shared__ __attribute__((aligned(16))) char s_state[sizeof(WaveState)];
    __shared__ uint32_t s_grid[kEncGrid / 4];
    WaveState &ps = *reinterpret_cast<WaveState *>(s_state);
    const int lane = threadIdx.x;
    const unsigned long long total = (unsigned long long)npos * nplay;
    ps.moves.rest = spill + (size_t)blockIdx.x * kSpillMoves;
    for (;;) {
        unsigned long long i = 0;
        if (lane == 0) i = atomicAdd(next, 1ull);
        i = (unsigned long long)__builtin_amdgcn_readfirstlane((uint32_t)i) |
            (unsigned long long)__builtin_amdgcn_readfirstlane(
                (uint32_t)(i >> 32))
                << 32;
        if (i >= total) return;
        const int p = (int)(i / nplay), j = (int)(i % nplay);
        const EncRecord &r = recs[p];
        for (int k = lane; k < kEncGrid / 4; k += 64)
            s_grid[k] = reinterpret_cast<const uint32_t *>(r.sq)[k];
        __syncthreads();
        ps.board.setup(r.side, reinterpret_cast<const uint8_t *>(s_grid));
        ps.to_move = r.to_move;
        ps.komove = r.komove;
        ps.last_move = r.last_move;
        ps.last_was_capture = r.last_was_capture != 0;
        ps.passes = r.passes;
        ps.movenum = r.movenum;
        ps.komi = r.komi;
        Rng rng(playout_seed(seed0 + (uint32_t)p, (uint32_t)j));
        rng.next();
        rng.next();
        const float score = ps.playout(rng, tables);
        if (lane == 0) {
            if (ps.overflow) {
                atomicAdd(&overflow[p], 1u);
            } else {
                const uint32_t h = score > 0.0f ? 2u : score == 0.0f ? 1u : 0u;
                if (h) atomicAdd(&half_wins[p], h);
            }
        }
        __syncthreads();
    }
}

// mc_owner's win rate for the side to move from the half-point counts,
// with the host's float operations; NaN for a position with an abandoned
// playout.
__global__ __launch_bounds__(64) void pat_winrate(
    const uint32_t *half_wins, const uint32_t *overflow,
    const EncRecord *recs, int npos, int nplay, float *winrate) {
    const int i = blockIdx.x * 64 + threadIdx.x;
    if (i >= npos) return;
    float w = nplay > 0 ? (float)half_wins[i] * 0.5f / (float)nplay : 0.5f;
    if (recs[i].to_move != mc::kBlack) w = 1.0f - w;
    winrate[i] = overflow[i] ? __builtin_nanf("") : w;
}

}  // namespace

size_t pattern_state_bytes() { return sizeof(mc::Move) * kSpillMoves; }

hipError_t launch_pattern_playouts(const EncRecord *d_rec, int npos,
                                   int nplay, uint32_t seed0,
                                   const mc::TablesView &tables,
                                   void *d_states, int nstates,
                                   unsigned long long *d_next,
                                   uint32_t *d_half_wins,
                                   uint32_t *d_overflow, float *d_winrate,
                                   hipStream_t stream) {
    if (npos <= 0) return hipSuccess;
    if (nstates < 1) return hipErrorInvalidValue;
    const int blocks = (npos + 63) / 64;
    hipLaunchKernelGGL(pat_zero, dim3(blocks), dim3(64), 0, stream,
                       d_half_wins, d_overflow, npos, d_next);
    const long long total = (long long)npos * nplay;
    if (total > 0) {
        const long long waves = total < nstates ? total : nstates;
        hipLaunchKernelGGL(pat_playout_kernel, dim3((unsigned)waves), dim3(64),
                           0, stream, d_rec, npos, nplay, seed0, tables,
                           static_cast<mc::Move *>(d_states), d_next,
                           d_half_wins, d_overflow);
    }
    hipLaunchKernelGGL(pat_winrate, dim3(blocks), dim3(64), 0, stream,
                       d_half_wins, d_overflow, d_rec, npos, nplay, d_winrate);
    return hipGetLastError();
}

}  // namespace lz
