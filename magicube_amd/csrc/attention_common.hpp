// Quantized sparse-attention building blocks shared by the fused batched
// kernel and the one-op-per-launch kernels, so both produce identical
// integers (int32 logits, int8 probabilities, int32 outputs).
//
// Layer semantics (end2end_eval/sparse_transformer_magicube/spattention.py:
// 182-216): per (sample, head) matrix with sequence length L and head dim 64,
//   S = Qq Kq^T at the vector-sparse mask          (int32, exact)
//   s = float(S) * alpha        alpha = 1 / (scale_q * scale_k * sqrt(64))
//   reference requantization (q_softmax_kernel.cu:132-147):
//     P = trunc(min(exp(s - max_row) / sum_row * scale_p, 127))   (int8 >= 0)
//     O = float(P Vq) * o_scale          o_scale = 1 / (scale_v * scale_p)
//   row-scaled requantization (full int8 range in every row, rounded):
//     P = rint(min(exp(s - max_row) * scale_p, 127))
//     O = (float(P Vq) * o_scale) * (1 / sum_row)
// Rows are the V matrix rows of one vector row; max/sum run over the row's
// nonzero slots.
//
// Canonical softmax statistics: the exact max m over the row; lane c of 16
// adds exp(s - m) of its slots chunk by chunk of 64 (four 16-slot MFMA tiles,
// slot order), (e0 + e1) + (e2 + e3) of the slots c, 16 + c, 32 + c, 48 + c of
// a chunk at a time, then the 16 lane sums are added as a pairwise tree over
// lane order.  Rows of more than kRowChunks chunks whose P needs the sum (the
// reference modes) are not visited a third time: there each lane keeps the
// sum against its own running max, rescaled when that grows, and brings it to
// the row max before the tree.  Both kernels evaluate these statistics on the
// same register layout (MFMA C layout: lane (c, g) holds rows 4g+i of
// slot 16t + c) with the same instructions.  The fused kernel deals the V
// real rows to the four 16-lane groups as it loads Q (tile rows 4q + j), so
// it keeps fewer rows per lane and moves none; each row is still held by the
// 16 lanes c of one group with slots 16t + c, and its statistics take the
// same operations in the same order.
#pragma once

#include <hip/hip_fp16.h>

#include "mc_device.hpp"
#include "mc_internal.hpp"

namespace mc {

// Device view of mc_attn_matrix (same member order and types).
struct AttnMatrix {
    int L;
    int m_vec;
    const int *row_offsets;
    const int *col_indices;
    const unsigned char *q;
    const unsigned char *k;
    const unsigned char *v;
    float alpha;
    float o_scale;
    float *o;
    int *o_int;
    unsigned char *p_out;
    int *s_out;
    __half *o16;
    int o16_stride;
    int o16_pad;
    const __half *q16;
    int q16_stride;
    float q_scale;
    int q_rounding;
    int q_pad;
};
static_assert(sizeof(AttnMatrix) == sizeof(mc_attn_matrix), "descriptor layout");

constexpr int kHeadDim = 64;

// Chunks of 64 slots whose logits the fused kernel holds: its LDS copy
// (kLogitStashBytes per wave: six chunks at V = 8, twelve at V = 2 and 4) and
// two more in registers.
constexpr int kLogitStashBytes = 12288;   // per wave
template <int V> constexpr int kStashChunks = kLogitStashBytes / (64 * 16 * (V == 8 ? 2 : 1));
template <int V> constexpr int kRowChunks = kStashChunks<V> + 2;

// Butterfly reductions within each 16-lane row of the wave, on DPP lane
// moves (no LDS round trip): swap neighbours, swap pairs (quad_perm), then
// combine the two quads of each 8-lane half (row_half_mirror) and the two
// halves (row_mirror).  Each step adds the same two partial results in every
// lane that holds them (in commuted order), so every lane of the row ends
// with the same bits, equal to the xor butterfly over lane distances 1, 2,
// 4, 8: ((x0+x1)+(x2+x3)) + ((x4+x5)+(x6+x7)) ... for a sum.
template <int CTRL> __device__ __forceinline__ float dpp_move(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, false));
}
constexpr int kDppSwap1 = 0xB1;        // quad_perm [1, 0, 3, 2]
constexpr int kDppSwap2 = 0x4E;        // quad_perm [2, 3, 0, 1]
constexpr int kDppHalfMirror = 0x141;  // lane i <- lane 7 - i within 8
constexpr int kDppMirror = 0x140;      // lane i <- lane 15 - i within 16
__device__ __forceinline__ float row16_max(float x) {
    x = fmaxf(x, dpp_move<kDppSwap1>(x));
    x = fmaxf(x, dpp_move<kDppSwap2>(x));
    x = fmaxf(x, dpp_move<kDppHalfMirror>(x));
    x = fmaxf(x, dpp_move<kDppMirror>(x));
    return x;
}
__device__ __forceinline__ float row16_sum(float x) {
    x = x + dpp_move<kDppSwap1>(x);
    x = x + dpp_move<kDppSwap2>(x);
    x = x + dpp_move<kDppHalfMirror>(x);
    x = x + dpp_move<kDppMirror>(x);
    return x;
}

// A logit scaled and rounded by itself: a following subtraction of the row
// max is never contracted with it, whichever way the value reaches it.
__device__ __forceinline__ float scaled_logit(int v, float alpha) {
#pragma clang fp contract(off)
    return (float)v * alpha;
}

// max of two values that are no NaN, in one instruction: fmaxf first quiets
// each input that comes through a branch or memory.
__device__ __forceinline__ float max2(float a, float b) { return __builtin_amdgcn_fmed3f(a, b, INFINITY); }

// s[t][i]: scaled logit of slot 16t + c for the lane's row i (-inf when masked).
template <int HOME, int W>
__device__ __forceinline__ void softmax_lane_max(const float (&s)[4][W], float (&m)[HOME]) {
    static_assert(HOME <= W, "rows held per lane");
#pragma unroll
    for (int i = 0; i < HOME; ++i) m[i] = max2(m[i], max2(max2(s[0][i], s[1][i]), max2(s[2][i], s[3][i])));
}
// exp(s - m) of one chunk in place (m finite; a masked slot gives exactly 0),
// and its part of the lane sums.
template <int HOME, int W>
__device__ __forceinline__ void softmax_lane_exp(float (&s)[4][W], const float (&m)[HOME], float (&l)[HOME]) {
#pragma unroll
    for (int i = 0; i < HOME; ++i) {
#pragma unroll
        for (int t = 0; t < 4; ++t) s[t][i] = __expf(s[t][i] - m[i]);
        l[i] += (s[0][i] + s[1][i]) + (s[2][i] + s[3][i]);
    }
}
// The lane's running max and its sum against that max after one chunk.  The
// offset is 0 while the lane has no slot yet (-inf - -inf would be NaN); its
// sum is 0 then.
template <int HOME, int W>
__device__ __forceinline__ void softmax_lane_update(const float (&s)[4][W], float (&m)[HOME], float (&l)[HOME]) {
#pragma unroll
    for (int i = 0; i < HOME; ++i) {
        const float mn = max2(m[i], max2(max2(s[0][i], s[1][i]), max2(s[2][i], s[3][i])));
        const float mz = mn == -INFINITY ? 0.f : mn;
        float e[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) e[t] = __expf(s[t][i] - mz);
        l[i] = l[i] * __expf(m[i] - mz) + ((e[0] + e[1]) + (e[2] + e[3]));
        m[i] = mn;
    }
}

constexpr int kPModeReference = 0;
constexpr int kPModeRowScaled = 1;
constexpr int kPModeReference4 = 2;   // reference requantization into 4-bit P

// Row max as quantize_prob takes it: 0 for a row without slots.
__device__ __forceinline__ float finite_row_max(float m) { return m == -INFINITY ? 0.f : m; }

// Quantized probability of one logit given the final row statistics
// (m from finite_row_max); a masked slot (s = -inf) gives exp(-inf) = 0.
__device__ __forceinline__ int quantize_prob(float s, float m, float inv_l, float p_scale, int p_mode) {
    const float e = __expf(s - m);
    if (p_mode != kPModeRowScaled)   // truncation (p >= 0)
        return (int)fminf(e * inv_l * p_scale, p_mode == kPModeReference4 ? 7.f : 127.f);
    return (int)rintf(fminf(e * p_scale, 127.f));
}
// The same value from the exponential, the mode fixed at compile time (the
// fused kernel's chunk loops), as the low byte of the result (the other bytes
// undefined).
// Without `clamp` (exponential and 1 / sum at most 1, p_scale at most 127) the
// value cannot exceed 127; adding 1.5 * 2^23 rounds to the nearest integer
// (ties to even, as rintf) and leaves it in the low bits.
template <int PM>
__device__ __forceinline__ u32 quantize_exp_byte(float e, float inv_l, float p_scale, bool clamp) {
    float t = PM == kPModeRowScaled ? e * p_scale : e * inv_l * p_scale;
    if (clamp) t = fminf(t, PM == kPModeReference4 ? 7.f : 127.f);
    if constexpr (PM == kPModeRowScaled) {
#pragma clang fp contract(off)
        return __float_as_uint(t + 12582912.f);
    }
    return (u32)(int)t;
}

// Moves P from the lanes' row layout (lane (c, g): rows row0 + i of slot
// 16t + c; row0 = 4g in the MFMA C layout) to the MFMA A layout (lane (r, g):
// row r, slots 16g..16g+15) through a per-wave 16 x 64 byte LDS tile laid
// out [row][slot].
template <int HOME, int W>
__device__ __forceinline__ v4i p_to_a_layout(unsigned char *tile, const int (&pq)[4][W], int lane, bool home,
                                             int row0) {
    static_assert(HOME <= W, "rows held per lane");
    const int c = lane & 15, g = lane >> 4;
    if (home) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < HOME; ++i) tile[(row0 + i) * 64 + 16 * t + c] = (unsigned char)pq[t][i];
    }
    // The tile is private to the wave and LDS operations of one wave complete
    // in order, so wavefront-scope fences (no waits) are enough: they keep
    // the compiler from moving the read above the writes (and the next writes
    // above this read).  Workgroup scope would also wait for every gather in
    // flight that lands in LDS.  Rows >= V are never written and only feed
    // output rows that are discarded.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const v4i a = *reinterpret_cast<const v4i *>(tile + c * 64 + 16 * g);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    return a;
}

// The same move with each lane's four slots 16t + c of a row packed in one
// dword (byte t), the lane's rows at tile rows 4g + i: lane (r, g) gets tile
// row r, byte b = slot 16 (b % 4) + 4g + b / 4.
// Two dword writes per lane (V = 8) instead of eight byte writes.
template <int HOME>
__device__ __forceinline__ v4i p_dwords_to_a_layout(unsigned char *tile, const u32 (&pq)[HOME], int lane, bool home) {
    const int c = lane & 15, g = lane >> 4;
    if (home) {
#pragma unroll
        for (int i = 0; i < HOME; ++i) *reinterpret_cast<u32 *>(tile + (4 * g + i) * 64 + 4 * c) = pq[i];
    }
    // wavefront-scope fences, as above
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const v4i a = *reinterpret_cast<const v4i *>(tile + c * 64 + 16 * g);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    return a;
}

}  // namespace mc
