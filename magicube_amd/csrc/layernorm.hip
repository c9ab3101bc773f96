// Row LayerNorm on fp16 activations for the encoder benchmark, optionally
// fused with the residual add before it:
//   s = half(x + residual)          (or s = x)
//   y = half((s - mean) * rstd * weight + bias),   rstd = 1 / sqrt(var + eps)
// with mean and the biased variance of s taken in fp32 over the row, as
// torch's nn.LayerNorm computes for fp16 input.  The reference's encoder uses
// torch's LayerNorm and a separate residual add
// (end2end_eval/sparse_transformer_magicube/end_to_end.py:77-89).
//
// A lane holds 8 (1024 columns: 16) consecutive values of a row, loaded and
// stored 16 bytes at a time, so that a row of 256 takes half a wave.  The row
// statistics are two reductions (sum, then sum of squared deviations): a
// two-pass variance of values held in registers.
//
// Bound by memory: 32768 rows of 256 take 8.3 us (4.0 TB/s; a copy of that
// size 6.5), with the residual 11.9.  Before, a lane held 4 values and read
// the weight and the bias two bytes at a time, eight loads beside two of x:
// 11.8 and 16.7 us; 16384 rows of 512 16.0 (now 8.2), 8192 of 1024 with the
// residual 30.6 (now 13.0).
#include <hip/hip_fp16.h>

#include "mc_internal.hpp"

namespace mc {
namespace {

// x + the value of the lane a DPP pattern names (within each row of 16 lanes)
#define LN_DPP_ADD(x, ctrl) \
    ((x) + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), (ctrl), 0xF, 0xF, false)))

// Sum over the LPR (32 or 64) lanes of a row, the same value in each of
// them: within each row of 16
// lanes by DPP (lane pairs 1 apart, 2 apart, then the half-row and row
// mirrors; each step adds the same two values in both lanes of a pair),
// then the four sums of 16 read with v_readlane.  No LDS traffic.
template <int LPR> __device__ __forceinline__ float ln_row_sum(float x) {
    x = LN_DPP_ADD(x, 0xB1);     // quad_perm [1, 0, 3, 2]
    x = LN_DPP_ADD(x, 0x4E);     // quad_perm [2, 3, 0, 1]
    x = LN_DPP_ADD(x, 0x141);    // row_half_mirror
    x = LN_DPP_ADD(x, 0x140);    // row_mirror
    const float r0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 0));
    const float r1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 16));
    const float r2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 32));
    const float r3 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 48));
    if constexpr (LPR == 32) return (threadIdx.x & 32) ? r2 + r3 : r0 + r1;
    return (r0 + r1) + (r2 + r3);
}

// 16 bytes at 8-byte (activations) and 2-byte (weight, bias) alignment
typedef int half8 __attribute__((ext_vector_type(4), aligned(8)));
typedef int half8_any __attribute__((ext_vector_type(4), aligned(2)));
__device__ __forceinline__ __half2 half_pair(int w) { return *reinterpret_cast<const __half2 *>(&w); }

// Loads of x per wave, all issued before the first reduction: two (four rows
// of 256) take 8.3 us for 32768 rows of 256, four 8.8, eight 9.6.
constexpr int kLoadsPerWave = 2;

template <int COLS> struct LnShape {
    static constexpr int LPR = COLS == 256 ? 32 : 64;        // lanes of a row
    static constexpr int VPL = COLS / LPR;                   // values per lane
    static constexpr int NQ = VPL / 8;                       // 16-byte pieces per lane
    static constexpr int R = kLoadsPerWave / NQ;             // rows a lane takes part in
    static constexpr int kRows = R * (64 / LPR);             // rows per wave
};

template <int COLS>
__global__ __launch_bounds__(256) void layernorm_f16_kernel(long long rows, const __half *x, const __half *res,
                                                            const __half *weight, const __half *bias, float eps,
                                                            __half *out) {
    using S = LnShape<COLS>;
    constexpr int LPR = S::LPR, VPL = S::VPL, NQ = S::NQ, R = S::R;
    const int lane = threadIdx.x & 63;
    const long long wave0 = ((long long)blockIdx.x * 4 + (threadIdx.x >> 6)) * S::kRows;   // wave-uniform
    if (wave0 >= rows) return;
    // row r of the lane: row0 + r * (64 / LPR); rows past the end repeat the last
    const long long row0 = wave0 + lane / LPR;
    const size_t col = (size_t)(lane % LPR) * VPL;
    const auto base = [&](int r) {
        const long long row = row0 + r * (64 / LPR);
        return (size_t)(row < rows ? row : rows - 1) * COLS + col;
    };
    half8 h[R][NQ], hr[R][NQ];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int q = 0; q < NQ; ++q) h[r][q] = *reinterpret_cast<const half8 *>(x + base(r) + 8 * q);
    if (res) {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int q = 0; q < NQ; ++q) hr[r][q] = *reinterpret_cast<const half8 *>(res + base(r) + 8 * q);
    }
    float wv[VPL], bv[VPL];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const half8_any one = {0x3C003C00, 0x3C003C00, 0x3C003C00, 0x3C003C00}, zero = {0, 0, 0, 0};
        const half8_any w8 = weight ? *reinterpret_cast<const half8_any *>(weight + col + 8 * q) : one;
        const half8_any b8 = bias ? *reinterpret_cast<const half8_any *>(bias + col + 8 * q) : zero;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            wv[8 * q + 2 * e] = __low2float(half_pair(w8[e]));
            wv[8 * q + 2 * e + 1] = __high2float(half_pair(w8[e]));
            bv[8 * q + 2 * e] = __low2float(half_pair(b8[e]));
            bv[8 * q + 2 * e + 1] = __high2float(half_pair(b8[e]));
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        float v[VPL];
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                __half2 a = half_pair(h[r][q][e]);
                if (res) a = __hadd2(a, half_pair(hr[r][q][e]));     // rounded to fp16, as a separate add would store it
                v[8 * q + 2 * e] = __low2float(a);
                v[8 * q + 2 * e + 1] = __high2float(a);
            }
        float sum = 0.f;
#pragma unroll
        for (int q = 0; q < VPL; ++q) sum += v[q];
        const float mean = ln_row_sum<LPR>(sum) * (1.0f / COLS);
        float sq = 0.f;
#pragma unroll
        for (int q = 0; q < VPL; ++q) {
            const float d = v[q] - mean;
            sq += d * d;
        }
        const float rstd = rsqrtf(ln_row_sum<LPR>(sq) * (1.0f / COLS) + eps);
        if (row0 + r * (64 / LPR) >= rows) continue;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            half8 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int i = 8 * q + 2 * e;
                const float y0 = (v[i] - mean) * rstd * wv[i] + bv[i];
                const float y1 = (v[i + 1] - mean) * rstd * wv[i + 1] + bv[i + 1];
                const __half2 y = __floats2half2_rn(y0, y1);
                o[e] = *reinterpret_cast<const int *>(&y);
            }
            *reinterpret_cast<half8 *>(out + base(r) + 8 * q) = o;
        }
    }
}

template <int COLS>
mc_status layernorm_launch(long long rows, const __half *x, const __half *res, const __half *weight, const __half *bias,
                           float eps, __half *out, hipStream_t stream) {
    constexpr int per_block = 4 * LnShape<COLS>::kRows;
    const long long blocks = (rows + per_block - 1) / per_block;
    if (blocks > 0x7FFFFFFFLL) return MC_EINVAL_SHAPE;
    hipLaunchKernelGGL((layernorm_f16_kernel<COLS>), dim3((unsigned)blocks), dim3(256), 0, stream, rows, x, res,
                       weight, bias, eps, out);
    return check_launch();
}

}  // namespace
}  // namespace mc

extern "C" {

mc_status mc_layernorm_f16(long long rows, int cols, const void *x, const void *residual, const void *weight,
                           const void *bias, float eps, void *out, hipStream_t stream) {
    if (rows < 0 || (cols != 256 && cols != 512 && cols != 1024)) return MC_EINVAL_SHAPE;
    if (rows == 0) return MC_OK;
    if (!x || !out) return MC_EINVAL_ARG;
    // vector loads and stores of 8-byte alignment
    const auto aligned = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 7u) == 0; };
    if (!aligned(x) || !aligned(out) || (residual && !aligned(residual))) return MC_EINVAL_ARG;
    const auto *px = static_cast<const __half *>(x);
    const auto *pr = static_cast<const __half *>(residual);
    const auto *pw = static_cast<const __half *>(weight);
    const auto *pb = static_cast<const __half *>(bias);
    auto *po = static_cast<__half *>(out);
    switch (cols) {
    case 256: return mc::layernorm_launch<256>(rows, px, pr, pw, pb, eps, po, stream);
    case 512: return mc::layernorm_launch<512>(rows, px, pr, pw, pb, eps, po, stream);
    default: return mc::layernorm_launch<1024>(rows, px, pr, pw, pb, eps, po, stream);
    }
}

}  // extern "C"
