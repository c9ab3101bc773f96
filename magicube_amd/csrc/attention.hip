// Quantized sparse attention on gfx950: quantize, softmax + requantize,
// dequantize, and the fused batched kernel (one wave per (matrix, vector row)
// work item, persistent over a longest-first work list), plus the C ABI.
#include <hip/hip_fp16.h>

#include <type_traits>

#include "attention_common.hpp"
#include "mc_internal.hpp"
#include "sddmm_kernel.hpp"

namespace mc {

// ---------------------------------------------------------------------------
// quantize: q = trunc(clamp(float(x) * scale, lo, hi)), or rint() for nearest
// (end2end_eval/sparse_transformer_magicube/src/cuda/quantization_kernel.cu:46-74
// for 8 bits, :13-43 for 4 bits; 4-bit lanes packed 8 per int32, lane 0 low)
// ---------------------------------------------------------------------------
struct QuantJob {
    const __half *x;
    long long count;
    float scale;
    void *out;
    long long row_len;      // 0: x is contiguous; else rows of row_len values,
    long long row_stride;   // row_stride values apart (row_len % 8 == 0)
};
static_assert(sizeof(QuantJob) == sizeof(mc_quant_job), "job layout");

// Groups of 8 consecutive values that one thread converts per pass: the
// block covers 256 * kQuantGroups groups, thread t takes groups t, t + 256,
// ... of them, and all of its loads are issued before any is converted.
constexpr int kQuantGroups = 2;

// the job's pointers come from memory: without the address space every access
// is a flat one, whose loads also wait for LDS
typedef __attribute__((address_space(1))) const v4i global_v4i;
typedef __attribute__((address_space(1))) v2i global_v2i;
typedef __attribute__((address_space(1))) u32 global_u32;

__device__ __forceinline__ void unpack_half8(const v4i &w, float (&x)[8]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int we = w[e];
        const __half2 h2 = *reinterpret_cast<const __half2 *>(&we);
        x[2 * e] = __low2float(h2);
        x[2 * e + 1] = __high2float(h2);
    }
}

// 8 values -> 8 int8 or packed int4 at group gi of the job's output
template <int BITS>
__device__ __forceinline__ void quantize_group(const float (&x)[8], const QuantJob &jb, int rounding, float lo,
                                               float hi, long long gi) {
    int q[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        float f = x[e] * jb.scale;
        f = fminf(fmaxf(f, lo), hi);
        q[e] = (rounding & 1) == 0 ? (int)f : (int)rintf(f);
    }
    if constexpr (BITS == 8) {
        unsigned char *o = static_cast<unsigned char *>(jb.out) + gi * 8;
        if (gi * 8 + 8 <= jb.count) {
            u32 w0 = (u32)(q[0] & 255) | (u32)(q[1] & 255) << 8 | (u32)(q[2] & 255) << 16 | (u32)(q[3] & 255) << 24;
            u32 w1 = (u32)(q[4] & 255) | (u32)(q[5] & 255) << 8 | (u32)(q[6] & 255) << 16 | (u32)(q[7] & 255) << 24;
            *(global_v2i *)o = v2i{(int)w0, (int)w1};
        } else {
            for (int e = 0; gi * 8 + e < jb.count; ++e) o[e] = (unsigned char)q[e];
        }
    } else {
        u32 wq = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) wq |= (u32)(q[e] & 15) << (4 * e);
        *((global_u32 *)jb.out + gi) = wq;
    }
}

template <int BITS> __device__ __forceinline__ void quantize_job(const QuantJob jb, int rounding) {
    // MC_QUANT_RANGE4 (bit 1 of rounding): 4-bit values in int8 storage
    const bool range4 = BITS == 4 || (rounding & 2) != 0;
    const float lo = range4 ? -8.f : -128.f, hi = range4 ? 7.f : 127.f;
    constexpr int G = kQuantGroups;
    const long long groups = (jb.count + 7) / 8;
    // Whole groups of a job whose rows start on 16 bytes and are 2^shift long
    // (every head dimension; shift 62: contiguous) take the branch-free loop:
    // clamped 16-byte loads, so that a thread's loads are in flight together.
    // Non-temporal: the fp16 source is read once, and keeping it out of the
    // caches leaves them to the quantized operands the fused kernel gathers
    // next.
    const bool regular = (jb.row_len & (jb.row_len - 1)) == 0 &&
                         (reinterpret_cast<uintptr_t>(jb.x) & 15u) == 0 && (jb.row_len == 0 || jb.row_stride % 8 == 0);
    long long done = 0;     // groups the first loop converts
    if (regular && jb.count >= 8) {
        const int shift = jb.row_len == 0 ? 62 : (int)__ffsll((unsigned long long)jb.row_len) - 1;
        const long long skip = jb.row_len == 0 ? 0 : jb.row_stride - jb.row_len;
        done = jb.count / 8;
        for (long long blk = blockIdx.x; blk * 256 * G < done; blk += gridDim.x) {
            const long long g0 = blk * 256 * G + threadIdx.x;
            v4i w[G];
#pragma unroll
            for (int k = 0; k < G; ++k) {
                const long long base = min(g0 + 256 * k, done - 1) * 8;
                w[k] = __builtin_nontemporal_load((global_v4i *)(jb.x + base + (base >> shift) * skip));
            }
#pragma unroll
            for (int k = 0; k < G; ++k) {
                float x[8];
                unpack_half8(w[k], x);
                if (g0 + 256 * k < done) quantize_group<BITS>(x, jb, rounding, lo, hi, g0 + 256 * k);
            }
        }
    }
    // the rest: the last part of a group, and jobs of other row lengths or
    // alignments (8 values never straddle a source row: row_len % 8 == 0), 16
    // bytes at a time where a group's source allows it: 32768 rows of 96 or 80
    // values take 4.5 us, value by value 5.8 and 5.6
    for (long long blk = blockIdx.x; done + blk * 256 * G < groups; blk += gridDim.x) {
        const long long g0 = done + blk * 256 * G + threadIdx.x;
        v4i w[G];
        const __half *src[G];
        bool vec[G];
#pragma unroll
        for (int k = 0; k < G; ++k) {
            const long long base = (g0 + 256 * k) * 8;
            src[k] = jb.row_len ? jb.x + (base / jb.row_len) * jb.row_stride + base % jb.row_len : jb.x + base;
            vec[k] = base + 8 <= jb.count && (reinterpret_cast<uintptr_t>(src[k]) & 15u) == 0;
            if (vec[k]) w[k] = __builtin_nontemporal_load((global_v4i *)src[k]);
        }
#pragma unroll
        for (int k = 0; k < G; ++k) {
            const long long gi = g0 + 256 * k;
            if (gi >= groups) continue;
            float x[8];
            if (vec[k]) {
                unpack_half8(w[k], x);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = gi * 8 + e < jb.count ? __half2float(src[k][e]) : 0.f;
            }
            quantize_group<BITS>(x, jb, rounding, lo, hi, gi);
        }
    }
}

// One job per blockIdx.y from a device array, or the one job passed as an
// argument (a single tensor: no descriptor to copy to the device first).
template <int BITS>
__global__ __launch_bounds__(256) void quantize_kernel(const QuantJob *jobs, int rounding) {
    const QuantJob job = jobs[blockIdx.y];       // a copy: stores to its output cannot change it
    quantize_job<BITS>(job, rounding);
}
template <int BITS> __global__ __launch_bounds__(256) void quantize_one_kernel(QuantJob job, int rounding) {
    quantize_job<BITS>(job, rounding);
}

// max |x| over a tensor, combined with atomicMax on the float bit pattern
// (non-negative floats order like their bits); *out must start at 0.
__global__ __launch_bounds__(256) void absmax_kernel(const __half *x, long long count, unsigned *out) {
    float m = 0.f;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < count; i += (long long)gridDim.x * 256)
        m = fmaxf(m, fabsf(__half2float(x[i])));
    for (int s = 32; s > 0; s >>= 1) m = fmaxf(m, __shfl_xor(m, s, 64));
    __shared__ float part[4];
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        const float b = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
        atomicMax(out, __float_as_uint(b));
    }
}

// dequantize: out[r][c] = (float(in[r][c]) * scale) * row_scale[r]  (row_scale optional)
__global__ __launch_bounds__(256) void dequant_kernel(const int *in, long long count, int cols, float scale,
                                                      const float *row_scale, float *out) {
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < count; i += (long long)gridDim.x * 256) {
        float f = (float)in[i] * scale;
        if (row_scale) f = f * row_scale[i / cols];
        out[i] = f;
    }
}

// ---------------------------------------------------------------------------
// softmax + requantize (q_softmax_kernel.cu:180-271): one wave per vector
// row.  S is int32 vector-major [slot][V] (the SDDMM output); P is written
// in the SpMM A layout: groups of 16 slots, [V][16] bytes per group.
// ---------------------------------------------------------------------------
template <int V, int WPB>
__global__ __launch_bounds__(64 * WPB) void softmax_requant_kernel(int m_vec, const int *row_indices,
                                                                   const int *row_offsets, const int *s_vals,
                                                                   float alpha, float p_scale, int p_mode,
                                                                   unsigned char *p_out, float *row_inv_l) {
    constexpr int HOME = V < 4 ? V : 4;
    __shared__ __attribute__((aligned(16))) unsigned char tiles[WPB][16 * 64];
    // the wave id in an SGPR keeps work-item indices, descriptors and buffer
    // resources wave-uniform (no per-lane waterfall around each buffer load)
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row_slot = blockIdx.x * WPB + wave;
    if (row_slot >= m_vec) return;
    const int c = lane & 15, g = lane >> 4;
    const bool home = g < (V + 3) / 4;
    const int i_row = uniform(row_indices ? row_indices[row_slot] : row_slot);
    const int start = uniform(row_offsets[2 * i_row]), end = uniform(row_offsets[2 * i_row + 1]);
    const int nch = (end - start + 63) >> 6;

    auto load_chunk = [&](int ch, float (&s)[4][4]) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int slot = start + 64 * ch + 16 * t + c;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int v = 4 * g + i;
                s[t][i] = (home && i < HOME && slot < end) ? scaled_logit(s_vals[(size_t)slot * V + v], alpha) : -INFINITY;
            }
        }
    };

    float m[HOME], l[HOME];
#pragma unroll
    for (int i = 0; i < HOME; ++i) { m[i] = -INFINITY; l[i] = 0.f; }
    float mq[HOME];
    const bool online = p_mode != kPModeRowScaled && nch > kRowChunks<V>;
    for (int ch = 0; ch < nch; ++ch) {
        float s[4][4];
        load_chunk(ch, s);
        if (online) softmax_lane_update<HOME>(s, m, l);
        else softmax_lane_max<HOME>(s, m);
    }
#pragma unroll
    for (int i = 0; i < HOME; ++i) mq[i] = finite_row_max(row16_max(m[i]));
    if (online) {
#pragma unroll
        for (int i = 0; i < HOME; ++i) l[i] *= __expf(m[i] - mq[i]);
    } else {
        for (int ch = 0; ch < nch; ++ch) {
            float s[4][4];
            load_chunk(ch, s);
            softmax_lane_exp<HOME>(s, mq, l);
        }
    }
#pragma unroll
    for (int i = 0; i < HOME; ++i) l[i] = row16_sum(l[i]);
    float inv_l[HOME];
#pragma unroll
    for (int i = 0; i < HOME; ++i) inv_l[i] = l[i] > 0.f ? 1.0f / l[i] : 0.f;
    if (row_inv_l && home && c == 0) {
#pragma unroll
        for (int i = 0; i < HOME; ++i) row_inv_l[(size_t)i_row * V + 4 * g + i] = inv_l[i];
    }
    // padded slots of the row (up to the next multiple of 16) get P = 0
    const int aend = start + ((end - start + 15) & ~15);
    const int nch_w = (aend - start + 63) >> 6;
    for (int ch = 0; ch < nch_w; ++ch) {
        float s[4][4];
        load_chunk(ch, s);
        int pq[4][4];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                pq[t][i] = i < HOME ? quantize_prob(s[t][i], mq[i < HOME ? i : 0], inv_l[i < HOME ? i : 0], p_scale, p_mode) : 0;
        const v4i a = p_to_a_layout<HOME>(tiles[wave], pq, lane, home, 4 * g);
        const int slot0 = start + 64 * ch + 16 * g;        // first slot of this lane's 16-slot group
        if (c < V && slot0 < aend)
            *reinterpret_cast<v4i *>(p_out + (size_t)(slot0 >> 4) * 16 * V + 16 * c) = a;
    }
}

// dequantize to fp16: out[i] = half(float(in[i]) / divisor), round to nearest
// even (the reference's epilogues, deq_spmm_kernel.cu:645-670 and
// sddmm_utils/output_tile.h:37-43: __float2half((float)acc / scale))
__global__ __launch_bounds__(256) void dequant_f16_kernel(const int *in, long long count, float divisor,
                                                          __half *out) {
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < count; i += (long long)gridDim.x * 256)
        out[i] = __float2half_rn((float)in[i] / divisor);
}

// ---------------------------------------------------------------------------
// The reference's batched quantized softmax on fp16 logits
// (q_softmax_kernel.cu:180-271, host :394-479): for matrix b of a batch
// sharing one mask and each vector row m = row_indices[x],
//   s = float(values[slot][v]) * sqrt_dk
//   max_v = max over the row's nonzeros of s, starting from -1e10 for v = 0
//           and from 0 for v >= 1 (the reference's register init sets only
//           element 0, :209)
//   sum_v = sum of exp(s - max_v)
//   P = (char / short) clamp(exp(s - max_v) / sum_v * scale, lo, hi)
// written at the reference's layouts (attn + start * V * bits / 8 bytes):
//   8-bit   [(i/16)][v][16] bytes
//   16-bit  [(i/16)][v][low 16 bytes][high 16 bytes]
//   4-bit   [(i/32)][v][16 bytes], byte j = slot 2j (low nibble) | 2j+1
// Every slot of [start, start + roundup(nonzeros, A)) is written (A = 32 for
// 4-bit P, else 16), padding slots with 0.  The sum runs in a fixed order:
// lane l adds slots l, l + 64, ..., then a butterfly over the 64 lanes.
// ---------------------------------------------------------------------------
// A slot's V fp16 logits, packed two to a register.
template <int V> struct HalfVec {
    u32 w[V / 2];
    __device__ __forceinline__ float at(int v) const {
        const __half2 h2 = *reinterpret_cast<const __half2 *>(&w[v >> 1]);
        return v & 1 ? __high2float(h2) : __low2float(h2);
    }
    // element-wise maximum (of a NaN and a number, the number)
    __device__ __forceinline__ void take_max(const HalfVec &o) {
#pragma unroll
        for (int k = 0; k < V / 2; ++k) {
            typedef _Float16 h2 __attribute__((ext_vector_type(2)));
            const h2 r = __builtin_elementwise_max(*reinterpret_cast<const h2 *>(&w[k]),
                                                   *reinterpret_cast<const h2 *>(&o.w[k]));
            w[k] = *reinterpret_cast<const u32 *>(&r);
        }
    }
};
template <int V> __device__ __forceinline__ HalfVec<V> load_half_vec(const __half *p) {
    HalfVec<V> x;
    if constexpr (V == 8) {
        const v4i t = *reinterpret_cast<const v4i *>(p);
#pragma unroll
        for (int e = 0; e < 4; ++e) x.w[e] = (u32)t[e];
    } else {
#pragma unroll
        for (int k = 0; k < V / 2; ++k) {
            const __half2 t{p[2 * k], p[2 * k + 1]};
            x.w[k] = *reinterpret_cast<const u32 *>(&t);
        }
    }
    return x;
}

// Butterflies over the wave without LDS: within each row of 16 lanes by DPP
// (row16_max / row16_sum), then v_permlane16_swap and v_permlane32_swap give
// every lane its own and its partner row's value.  The sum adds the same
// pairs as the xor butterfly over lane distances 1, 2, 4, 8, 16, 32.
__device__ __forceinline__ float wave_max(float x) {
    x = row16_max(x);
    auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
__device__ __forceinline__ float wave_sum(float x) {
    x = row16_sum(x);
    auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}

// 4 x 4 byte transpose within each quad of lanes: lane q gets byte q of its
// quad's four dwords (lane k's as byte k).
__device__ __forceinline__ u32 quad_bytes(u32 x, u32 sel) {
    const u32 d0 = (u32)__builtin_amdgcn_update_dpp(0, (int)x, 0x00, 0xF, 0xF, false);
    const u32 d1 = (u32)__builtin_amdgcn_update_dpp(0, (int)x, 0x55, 0xF, 0xF, false);
    const u32 d2 = (u32)__builtin_amdgcn_update_dpp(0, (int)x, 0xAA, 0xF, 0xF, false);
    const u32 d3 = (u32)__builtin_amdgcn_update_dpp(0, (int)x, 0xFF, 0xF, 0xF, false);
    return perm(perm(d3, d2, sel), perm(d1, d0, sel), 0x05040100u);
}

// One wave per (vector row, matrix); lane l holds slots l, l + 64, ...  Bound
// by its instructions (13 million logits, three passes), so: the logits of a
// row's first NC chunks are read once and their exponentials kept in
// registers (rows beyond that are read again), the division by the row sum
// is a host-free corrected reciprocal (quotient_fast: the IEEE quotient)
// while the sum and scale lie within 2^40 of 1, wave reductions use no LDS,
// and each quad of lanes transposes its four slots' bytes, so that a row's
// four slots go out as one dword instead of four bytes.
template <int V, int BITS, int WPB>
__global__ __launch_bounds__(64 * WPB) void ref_softmax_kernel(int rows, const int *row_indices, const int *row_offsets,
                                                               const __half *values, long long values_stride,
                                                               float sqrt_dk, float scale, unsigned char *attn,
                                                               long long attn_stride) {
    constexpr int NC = V == 8 ? 8 : 16;          // chunks of 64 slots held in registers
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = blockIdx.x * WPB + wave;
    if (x >= rows) return;
    const long long b = blockIdx.y;
    const int m = uniform(row_indices ? row_indices[x] : x);
    const int start = uniform(row_offsets[2 * m]), nz = uniform(row_offsets[2 * m + 1]) - start;
    if (nz <= 0) return;                         // no slot to write
    const __half *val = values + b * values_stride + (size_t)start * V;
    unsigned char *out = attn + b * attn_stride + (size_t)start * V * BITS / 8;

    HalfVec<V> h[NC];                            // logits
    float s[NC][V];                              // their exponentials
    float mx[V], sm[V];
#pragma unroll
    for (int v = 0; v < V; ++v) { mx[v] = v == 0 ? -1e10f : 0.f; sm[v] = 0.f; }
    // lanes past the end repeat the last slot: it changes no maximum
#pragma unroll
    for (int c = 0; c < NC; ++c)
        if (64 * c < nz) h[c] = load_half_vec<V>(val + (size_t)min(64 * c + lane, nz - 1) * V);
    const auto scaled_max = [&](const HalfVec<V> &t) {
#pragma unroll
        for (int v = 0; v < V; ++v) mx[v] = fmaxf(mx[v], t.at(v) * sqrt_dk);
    };
    // the maximum over logits first, scaled once: rounding keeps order, so
    // for a positive factor it is the maximum of the scaled logits
    if (sqrt_dk > 0.f) {
        HalfVec<V> hm = h[0];
#pragma unroll
        for (int c = 1; c < NC; ++c)
            if (64 * c < nz) hm.take_max(h[c]);
        scaled_max(hm);
    } else {
#pragma unroll
        for (int c = 0; c < NC; ++c)
            if (64 * c < nz) scaled_max(h[c]);
    }
    for (int i = 64 * NC + lane; i < nz; i += 64) scaled_max(load_half_vec<V>(val + (size_t)i * V));
#pragma unroll
    for (int v = 0; v < V; ++v) mx[v] = wave_max(mx[v]);
    const auto expo = [&](float t, int v) { return __expf(__builtin_fmaf(t, sqrt_dk, -mx[v])); };
#pragma unroll
    for (int c = 0; c < NC; ++c)
        if (64 * c < nz) {
#pragma unroll
            for (int v = 0; v < V; ++v) s[c][v] = expo(h[c].at(v), v);
            if (64 * c + 64 > nz) {
                const bool in = 64 * c + lane < nz;
#pragma unroll
                for (int v = 0; v < V; ++v) s[c][v] = in ? s[c][v] : 0.f;
            }
#pragma unroll
            for (int v = 0; v < V; ++v) sm[v] += s[c][v];
        }
    for (int i = 64 * NC + lane; i < nz; i += 64) {
        const HalfVec<V> t = load_half_vec<V>(val + (size_t)i * V);
#pragma unroll
        for (int v = 0; v < V; ++v) sm[v] += expo(t.at(v), v);
    }
    // fast: every quotient this row can give an integer from stays in the
    // corrected reciprocal's range (an exponential below 2^-100 gives 0 with
    // either division), and 0 <= exponential / sum * scale <= hi needs no
    // clamp.  The sums are the same in every lane.
    constexpr float lo = BITS == 4 ? -8.f : BITS == 8 ? -128.f : -32768.f;
    constexpr float hi = BITS == 4 ? 7.f : BITS == 8 ? 127.f : 32767.f;
    float y[V];
    bool fast = scale >= 0.f && scale <= hi;
#pragma unroll
    for (int v = 0; v < V; ++v) {
        sm[v] = wave_sum(sm[v]);
        y[v] = 1.0f / sm[v];
        fast &= sm[v] >= 0x1p-40f && sm[v] <= 0x1p40f;
    }
    fast = __builtin_amdgcn_readfirstlane(fast) != 0;

    const int q = lane & 3;
    const u32 sel = (u32)q | (u32)(4 + q) << 8 | 0x0C0C0000u;
    const bool aligned = (reinterpret_cast<uintptr_t>(out) & 3) == 0;
    const auto store4 = [&](unsigned char *o, u32 w) {
        if (aligned) *reinterpret_cast<u32 *>(o) = w;
        else
            for (int k = 0; k < 4; ++k) o[k] = (unsigned char)(w >> (8 * k));
    };
    // P of the lane's slot 64c + lane from its exponentials; every slot of a
    // quad is written or none (rows are padded to 16 or 32 slots with 0)
    const int nw = BITS == 4 ? (nz + 31) & ~31 : (nz + 15) & ~15;
    const auto write = [&](auto quick, int c, const float (&e)[V]) {
        const int i = 64 * c + lane;
        u32 p[V < 4 ? 4 : V];
        if constexpr (V < 4) p[2] = p[3] = 0;
#pragma unroll
        for (int v = 0; v < V; ++v) {
            if constexpr (decltype(quick)::value) {
                p[v] = (u32)(int)(quotient_fast(e[v], sm[v], y[v]) * scale);
            } else {
                const float cl = fminf(fmaxf(e[v] / sm[v] * scale, lo), hi);
                p[v] = i < nz ? (u32)(int)cl : 0u;
            }
        }
        if (i >= nw) return;
#pragma unroll
        for (int h = 0; h < V; h += 4) {
            // rows h .. h + 3: lane q of the quad stores row h + q of its four slots
            const int row = h + q;
            const u32 w0 = (p[h] & 255) | (p[h + 1] & 255) << 8 | (p[h + 2] & 255) << 16 | p[h + 3] << 24;
            if constexpr (BITS == 4) {
                const u32 t = quad_bytes(w0 & 0x0F0F0F0Fu, sel);
                const u32 y2 = t | t >> 4;
                unsigned char *o = out + (size_t)(i >> 5) * V * 16 + 16 * row + ((i & 31) >> 2) * 2;
                if (row < V) {
                    if (aligned) *reinterpret_cast<unsigned short *>(o) = (unsigned short)perm(y2, y2, 0x0C0C0200u);
                    else { o[0] = (unsigned char)y2; o[1] = (unsigned char)(y2 >> 16); }
                }
            } else {
                unsigned char *o = out + (size_t)(i >> 4) * V * (2 * BITS) + 2 * BITS * row + ((i & 15) >> 2) * 4;
                const u32 t = quad_bytes(w0, sel);
                if (row < V) store4(o, t);
                if constexpr (BITS == 16) {
                    const u32 w1 = (p[h] >> 8 & 255) | (p[h + 1] >> 8 & 255) << 8 | (p[h + 2] >> 8 & 255) << 16 |
                                   p[h + 3] >> 8 << 24;
                    const u32 t1 = quad_bytes(w1, sel);
                    if (row < V) store4(o + 16, t1);
                }
            }
        }
    };
    const auto write_row = [&](auto quick) {
#pragma unroll
        for (int c = 0; c < NC; ++c)
            if (64 * c < nw) write(quick, c, s[c]);
        for (int c = NC; 64 * c < nw; ++c) {
            const HalfVec<V> t = load_half_vec<V>(val + (size_t)min(64 * c + lane, nz - 1) * V);
            float e[V];
#pragma unroll
            for (int v = 0; v < V; ++v) e[v] = 64 * c + lane < nz ? expo(t.at(v), v) : 0.f;
            write(quick, c, e);
        }
    };
    if (fast) write_row(std::true_type{});
    else write_row(std::false_type{});
}

// Row bounds are read-only for the whole launch; read through the constant
// address space at a wave-uniform address they become scalar loads (scalar
// cache, lgkmcnt), which neither wait behind nor hold back vector gathers.
__device__ __forceinline__ int const_load(const int *p) {
    typedef const __attribute__((address_space(4))) int const_int;
    return *(const const_int *)p;
}

// ---------------------------------------------------------------------------
// Fused batched attention: persistent waves walk a work list of (matrix,
// vector row) items.  Pass 1 gathers K rows, computes the int32 logits with
// MFMA and keeps the row maxima; pass 2 quantizes P from one exponential per
// logit, moves it to the A layout through LDS, gathers V rows (4x4 byte
// transposes) and accumulates O = P V with MFMA.
// VB = 4: V rows are packed 4-bit ([L][32] bytes, lane 0 low); each lane
// gathers the 16 bits of its four columns and widens them to the bytes
// V + 8 (0..15), so the MFMA forms P (V + 8) and 8 * (row sum of P) comes off
// the accumulators at the end (exact mod 2^32).
//
// Bound by the address and data path of L1 with VALU issue close behind, not by
// L2: sending every gather to one 4 KB window takes the same time, dropping the
// arithmetic or the gathers does not.  Counters: TD busy 89 % of the time (36 %
// of that waiting for L2), TA 78, VALU 69, LDS 36 over 128 matrices of L up to
// 4096, row-scaled P; 81, 68, 67 and 42 % over 32 of L = 4096, reference P.  So each logit is scaled, exponentiated and summed once: pass 1 needs
// the max alone, its logits go to pass 2 through LDS (the first SST chunks)
// and registers (two more); lanes keep their own sums, reduced once per row;
// the real rows sit in all four lane groups of the MFMA tile; four P bytes are
// written as one dword; K rows are gathered row-contiguous.  Measured, us per
// launch, before (online softmax per chunk in pass 1, K and P recomputed) and
// now: 32 matrices of L = 4096, 90 % sparse, V = 8, reference P 96 -> 80;
// 64 of L ~ U[512, 4096], row-scaled P 84 -> 70; 4 of L = 8192, 80 % sparse
// 163 -> 145; 16 of L = 4096, 80 % sparse, V = 2 243 -> 204.
// ---------------------------------------------------------------------------
// DBG instantiations also write the optional int32 S, int8 P and int32 P V
// outputs; the production ones carry no stores inside the chunk loops (a
// conditional store there would make every load wait drain the queue).
// LDS: 12 KB of logits and a 1 KB P tile per wave, 52 KB per workgroup, so
// three workgroups (three waves per SIMD, at most 168 registers) fit a CU's
// 160 KB.
template <int V, int QKB, int VB, int PM, int WPB, bool DBG>
__global__ __launch_bounds__(64 * WPB) __attribute__((amdgpu_waves_per_eu(3))) void attention_kernel(
    const AttnMatrix *mats, const int2 *items, int n_items, float p_scale) {
    constexpr int QROW = kHeadDim * QKB / 8;          // bytes per Q/K row
    constexpr int KCB = QROW / 4;                     // bytes of a K row per lane
    __shared__ __attribute__((aligned(16))) unsigned char tiles[WPB][16 * 64];
    // logits s[t][j] of a row's first SST chunks, kept from pass 1 for pass 2
    // (per wave; SQ 16-byte slots per lane, lane-major, so the accesses are
    // conflict-free)
    constexpr int SQ = V == 8 ? 2 : 1;            // 4 * HC floats per lane
    constexpr int SST = kStashChunks<V>;
    __shared__ v4f sstash[WPB][SST][SQ][64];
    // the wave id in an SGPR keeps work-item indices, descriptors and buffer
    // resources wave-uniform (no per-lane waterfall around each buffer load)
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15, g = lane >> 4;
    // The V rows sit in the MFMA's row tile at rows 4q + j, j < HC: lane group
    // g of the C tile then holds vector rows HC * g + j in its first HC
    // accumulators, so that the per-logit work and the epilogue run on real
    // rows in every lane without moving any (rows 0..V-1 would leave them in
    // half the lanes at V = 8 and a quarter at V = 4).  The other tile rows
    // read Q and P out of range or unwritten and feed nothing.
    constexpr int HC = V == 8 ? 2 : 1;
    constexpr int NCH = kRowChunks<V>;
    const bool chome = HC * g < V;
    const int row0 = HC * g;                                  // lane's vector rows row0 + j
    const int a_row = HC * (c >> 2) + (c & 3);                // vector row of tile row c
    const bool a_live = (c & 3) < HC && a_row < V;
    const int nwaves = gridDim.x * WPB;

    for (int it = blockIdx.x * WPB + wave; it < n_items; it += nwaves) {
        const int2 item = items[it];
        if (uniform(item.x) < 0) continue;           // padding slot of the work list
        const AttnMatrix Mv = mats[uniform(item.x)];
        AttnMatrix M;
        M.L = uniform(Mv.L);
        M.m_vec = uniform(Mv.m_vec);
        M.row_offsets = uniform(Mv.row_offsets);
        M.col_indices = uniform(Mv.col_indices);
        M.q = uniform(Mv.q);
        M.k = uniform(Mv.k);
        M.v = uniform(Mv.v);
        M.alpha = uniform(Mv.alpha);
        M.o_scale = uniform(Mv.o_scale);
        M.o = uniform(Mv.o);
        M.o_int = uniform(Mv.o_int);
        M.p_out = uniform(Mv.p_out);
        M.s_out = uniform(Mv.s_out);
        M.o16 = uniform(Mv.o16);
        M.o16_stride = uniform(Mv.o16_stride);
        M.q16 = uniform(Mv.q16);
        M.q16_stride = uniform(Mv.q16_stride);
        M.q_scale = uniform(Mv.q_scale);
        M.q_rounding = uniform(Mv.q_rounding);
        const int i_row = uniform(item.y);
        const int start = uniform(const_load(M.row_offsets + 2 * i_row)),
                  end = uniform(const_load(M.row_offsets + 2 * i_row + 1));
        const int aend = start + ((end - start + 15) & ~15);
        const int nch = (end - start + 63) >> 6;
        const u32 kv_bytes = (u32)M.L * QROW;
        const __amdgpu_buffer_rsrc_t rk = make_rsrc(M.k, kv_bytes);
        const __amdgpu_buffer_rsrc_t rv = make_rsrc(M.v, (u32)M.L * (kHeadDim * VB / 8));
        const __amdgpu_buffer_rsrc_t rq = make_rsrc(M.q, kv_bytes);

        // SDDMM A operand: Q rows of this vector row (rows >= V read out of range -> 0)
        v4i qop = v4i{0, 0, 0, 0};
        // fp16 Q (q16 non-null): lane (c, g) loads columns 16g .. 16g + 15
        // of row i_row * V + c here and quantizes them once the pipeline's
        // first index and K loads are out (quantize_q16)
        v4i qh0 = v4i{0, 0, 0, 0}, qh1 = v4i{0, 0, 0, 0};
        if (M.q16) {
            const __amdgpu_buffer_rsrc_t rq16 =
                make_rsrc(M.q16, (u32)(((u32)(M.L - 1) * (u32)M.q16_stride + kHeadDim) * 2u));
            const u32 off = a_live ? ((u32)(i_row * V + a_row) * (u32)M.q16_stride + (u32)(16 * g)) * 2u : 0x80000000u;
            qh0 = buf_load_b128(rq16, off);
            qh1 = buf_load_b128(rq16, off + 16u);
        } else {
            const u32 off = a_live ? (u32)(i_row * V + a_row) * QROW + (u32)(16 * g * QKB / 8) : 0x80000000u;
            qop = load_k16<QKB>(rq, off);
            if constexpr (QKB == 4) qop = expand_nibbles(qop, true, 0u);
        }
        // the quantize launch's expression (quantize_kernel), laid out as the
        // quantized operand would arrive: in order for int8; for int4 in
        // expand_nibbles' order (even, then odd columns of each 8)
        auto quantize_q16 = [&]() {
            const bool range4 = QKB == 4 || (M.q_rounding & 2) != 0;
            const float lo = range4 ? -8.f : -128.f, hi = range4 ? 7.f : 127.f;
            u32 qb[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int w = e < 8 ? qh0[e >> 1] : qh1[(e - 8) >> 1];
                const __half2 h2 = *reinterpret_cast<const __half2 *>(&w);
                float f = ((e & 1) ? __high2float(h2) : __low2float(h2)) * M.q_scale;
                f = fminf(fmaxf(f, lo), hi);
                qb[e] = (u32)((M.q_rounding & 1) == 0 ? (int)f : (int)rintf(f)) & 255u;
            }
            const auto pack = [&](int a, int b, int c2, int d) {
                return (int)(qb[a] | qb[b] << 8 | qb[c2] << 16 | qb[d] << 24);
            };
            if constexpr (QKB == 8) qop = v4i{pack(0, 1, 2, 3), pack(4, 5, 6, 7), pack(8, 9, 10, 11), pack(12, 13, 14, 15)};
            else qop = v4i{pack(0, 2, 4, 6), pack(1, 3, 5, 7), pack(8, 10, 12, 14), pack(9, 11, 13, 15)};
        };

        const __amdgpu_buffer_rsrc_t rc = make_rsrc(M.col_indices, 0x7FFFFFFFu);
        constexpr u32 kRowOob = 0x80000000u;
        // ---- the row.  The first SST chunks' logits are kept in LDS, and two
        // more in registers where that is the whole row (nch <= NCH): then K
        // is gathered once, the max and sum are reduced across lanes once and
        // every exponential is taken once.  Later chunks of longer rows are
        // gathered and multiplied again for their P.  Slot order: lane
        // 16g + p of an index load holds slot 16 (p % 4) + 4g + p / 4 of its
        // chunk, so that P packs four slots 16t + c per dword (t the byte) on
        // its way to the A layout while V offsets still come from the lane's
        // own row of 16.
        // Per half step for chunk ch: the index load of chunk ch + 2 and the
        // row gathers of chunk ch + 1 go out before chunk ch is consumed.
        // Loads retire in order, so each consumer waits only for older loads.
        const bool kept = nch <= NCH;
        const int pslot = 16 * (lane & 3) + 4 * g + ((lane >> 2) & 3);
        const int perm_addr = 4 * (4 * c + g);
        // per lane: byte offset of its slot's V row (index * 64), or the
        // out-of-range marker for slots past the row end (L * 64 < 2^31)
        auto load_idx = [&](int ch) {
            const int slot = start + 64 * ch + pslot;
            const u32 v = buf_load_b32(rc, slot < end ? (u32)slot * 4u : kRowOob);
            return slot < end ? v * (u32)kHeadDim : kRowOob;
        };
        // K rows of a tile, row-contiguous: lane 4i + j holds piece j of slot
        // 16t + i's row (16 L1 accesses for 16 rows; gathered in the operand
        // layout, 16 rows per 16 lanes, a load makes 64).  The row offset is
        // lane t of the lane's quad.  logits() moves the data to the operand
        // layout with one ds_bpermute per dword.
        auto load_krows = [&](u32 my_off, v4i (&kop)[4]) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                u32 row = (u32)quad_bcast((int)my_off, t);
                if constexpr (QKB == 4) row = (row >> 1) | (row & kRowOob);   // 32-byte rows, marker kept
                kop[t] = load_k16<QKB>(rk, row + (u32)(KCB * (lane & 3)));
            }
        };
        auto put = [&](int ch, const float (&s)[4][HC]) {
#pragma unroll
            for (int q = 0; q < SQ; ++q) {
                v4f x;
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = s[(4 * q + e) / HC][(4 * q + e) % HC];
                sstash[wave][ch][q][lane] = x;
            }
        };
        auto get = [&](int ch, float (&s)[4][HC]) {
#pragma unroll
            for (int q = 0; q < SQ; ++q) {
                const v4f x = sstash[wave][ch][q][lane];
#pragma unroll
                for (int e = 0; e < 4; ++e) s[(4 * q + e) / HC][(4 * q + e) % HC] = x[e];
            }
        };
        // scaled logits of one chunk
        auto logits = [&](int ch, const v4i (&kop)[4], float (&s)[4][HC]) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                v4i kk = row_to_operand<QKB == 4 ? 2 : 4>(kop[t], perm_addr);
                if constexpr (QKB == 4) kk = expand_nibbles(kk, true, 0u);
                const v4i acc = mfma_i8(qop, kk, v4i{0, 0, 0, 0});
                if constexpr (DBG) {
                    const int slot = start + 64 * ch + 16 * t + c;
                    if (M.s_out && chome && slot < end) {
#pragma unroll
                        for (int j = 0; j < HC; ++j) M.s_out[(size_t)slot * V + row0 + j] = acc[j];
                    }
                }
#pragma unroll
                for (int j = 0; j < HC; ++j) s[t][j] = scaled_logit(acc[j], M.alpha);
            }
            if (ch >= nch - 1) {     // only the row's last chunk has masked slots
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int j = 0; j < HC; ++j) s[t][j] = start + 64 * ch + 16 * t + c < end ? s[t][j] : -INFINITY;
            }
        };
        float m[HC], l[HC], inv_l[HC], mq[HC];
#pragma unroll
        for (int j = 0; j < HC; ++j) { m[j] = -INFINITY; l[j] = 0.f; inv_l[j] = 0.f; }
        // the running statistics after one chunk's logits
        auto update = [&](const float (&s)[4][HC]) {
            if (PM != kPModeRowScaled && !kept) softmax_lane_update<HC>(s, m, l);
            else softmax_lane_max<HC>(s, m);
        };
        float sreg[2][4][HC];
        const u32 off0 = load_idx(0), off1 = load_idx(1);
        u32 ia = off0, ib = off1;
        {
            v4i ka[4], kb[4];
            float s[4][HC];
            load_krows(ia, ka);
            if (M.q16) quantize_q16();
            for (int ch = 0; ch < SST; ch += 2) {
                if (ch >= nch) break;
                ia = load_idx(ch + 2);
                load_krows(ib, kb);
                logits(ch, ka, s);
                put(ch, s);
                update(s);
                __builtin_amdgcn_sched_barrier(0);
                if (ch + 1 >= nch) break;
                ib = load_idx(ch + 3);
                load_krows(ia, ka);
                logits(ch + 1, kb, s);
                put(ch + 1, s);
                update(s);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (nch > SST) {
                if (kept) {
                    load_krows(ib, kb);
                    logits(SST, ka, sreg[0]);
                    softmax_lane_max<HC>(sreg[0], m);
                    logits(SST + 1, kb, sreg[1]);
                    softmax_lane_max<HC>(sreg[1], m);
                } else {
                    for (int ch = SST; ch < nch; ch += 2) {
                        ia = load_idx(ch + 2);
                        load_krows(ib, kb);
                        logits(ch, ka, s);
                        update(s);
                        __builtin_amdgcn_sched_barrier(0);
                        ib = load_idx(ch + 3);
                        load_krows(ia, ka);
                        logits(ch + 1, kb, s);
                        update(s);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        }
        // V rows of slots in pslot order: lane 16g + p of the index load holds
        // byte p of the lane group's A operand; columns 4c..4c+3: dword c of an
        // int8 row, or the 16 bits at byte 2c of a packed 4-bit row
        auto load_vrows = [&](u32 my_off, u32 (&raw)[16]) {
#pragma unroll
            for (int p = 0; p < 16; ++p) {
                u32 row = (u32)row_bcast16((int)my_off, p);   // lane 16g + p
                if constexpr (VB == 4) {
                    row = (row >> 1) | (row & kRowOob);   // 32-byte rows, marker kept
                    raw[p] = buf_load_u16(rv, row + 2u * c);
                } else {
                    raw[p] = buf_load_b32(rv, row + 4u * c);
                }
            }
        };
        // V of the first chunk is in flight while the statistics finish
        ib = off1;
        u32 va[16], vb[16];
        load_vrows(off0, va);
#pragma unroll
        for (int j = 0; j < HC; ++j) mq[j] = finite_row_max(row16_max(m[j]));
        if constexpr (PM != kPModeRowScaled) {
            // P needs the row sum
            if (kept) {
                for (int ch = 0; ch < SST; ++ch) {
                    if (ch >= nch) break;
                    float s[4][HC];
                    get(ch, s);
                    softmax_lane_exp<HC>(s, mq, l);
                    put(ch, s);
                }
                if (nch > SST) {
                    softmax_lane_exp<HC>(sreg[0], mq, l);
                    softmax_lane_exp<HC>(sreg[1], mq, l);
                }
            } else {
#pragma unroll
                for (int j = 0; j < HC; ++j) l[j] *= __expf(m[j] - mq[j]);
            }
#pragma unroll
            for (int j = 0; j < HC; ++j) {
                l[j] = row16_sum(l[j]);
                inv_l[j] = l[j] > 0.f ? 1.0f / l[j] : 0.f;
            }
        }
        v4i oacc[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) oacc[b] = v4i{0, 0, 0, 0};
        int psum = 0;   // VB = 4: sum of P row c over this lane's slots of every chunk
        // exponentials and 1 / sum are at most 1: only a scale above 127 (or the
        // 4-bit mode) can exceed P's range
        const bool clamp = PM == kPModeReference4 || p_scale > 127.f;
        // O += P V of one chunk; s: its logits, or (reference modes, kept
        // rows) its exponentials
        auto output = [&](int ch, float (&s)[4][HC], const u32 (&raw_in)[16]) {
            if constexpr (PM == kPModeRowScaled) {
                softmax_lane_exp<HC>(s, mq, l);
            } else {
                if (!kept) {
#pragma unroll
                    for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int j = 0; j < HC; ++j) s[t][j] = __expf(s[t][j] - mq[j]);
                }
            }
            u32 pq[HC];
#pragma unroll
            for (int j = 0; j < HC; ++j) {
                u32 b[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) b[t] = quantize_exp_byte<PM>(s[t][j], inv_l[j], p_scale, clamp);
                pq[j] = perm(perm(b[3], b[2], 0x0C0C0400u), perm(b[1], b[0], 0x0C0C0400u), 0x05040100u);
            }
            const v4i pop = p_dwords_to_a_layout<HC>(tiles[wave], pq, lane, chome);
            if (DBG && M.p_out && a_live) {
                // byte b of the lane: row a_row, slot 16 (b % 4) + 4g + b / 4
#pragma unroll
                for (int b = 0; b < 16; ++b) {
                    const int slot = start + 64 * ch + 16 * (b & 3) + 4 * g + (b >> 2);
                    if (slot < aend)
                        M.p_out[(size_t)(slot >> 4) * 16 * V + 16 * a_row + (slot & 15)] =
                            (unsigned char)((u32)pop[b >> 2] >> (8 * (b & 3)));
                }
            }
            u32 raw[16];
#pragma unroll
            for (int p = 0; p < 16; ++p) {
                if constexpr (VB == 4) {
                    // nibbles n0..n3 of V -> bytes n0 + 8 .. n3 + 8
                    const u32 x = raw_in[p] ^ 0x8888u;
                    raw[p] = perm((x >> 4) & 0x0F0Fu, x & 0x0F0Fu, 0x05010400u);
                } else {
                    raw[p] = raw_in[p];
                }
            }
            if constexpr (VB == 4) psum += sum_bytes(pop);
            // after the 4x4 byte transposes, tr[q][b] holds column 4c + b of rows 4q..4q+3
            u32 tr[4][4];
#pragma unroll
            for (int q = 0; q < 4; ++q) transpose4x4(raw[4 * q], raw[4 * q + 1], raw[4 * q + 2], raw[4 * q + 3], tr[q]);
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const v4i bop = v4i{(int)tr[0][b], (int)tr[1][b], (int)tr[2][b], (int)tr[3][b]};
                oacc[b] = mfma_i8(pop, bop, oacc[b]);
            }
        };
        {
            float s[4][HC];
            for (int ch = 0; ch < SST; ch += 2) {
                if (ch >= nch) break;
                ia = load_idx(ch + 2);
                load_vrows(ib, vb);
                get(ch, s);
                output(ch, s, va);
                __builtin_amdgcn_sched_barrier(0);
                if (ch + 1 >= nch) break;
                ib = load_idx(ch + 3);
                load_vrows(ia, va);
                get(ch + 1, s);
                output(ch + 1, s, vb);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (nch > SST) {
                if (kept) {
                    load_vrows(ib, vb);
                    output(SST, sreg[0], va);
                    output(SST + 1, sreg[1], vb);
                } else {
                    // ia, ib: chunks SST and SST + 1; va: chunk SST
                    v4i ka[4], kb[4];
                    load_krows(ia, ka);
                    for (int ch = SST; ch < nch; ch += 2) {
                        ia = load_idx(ch + 2);
                        load_krows(ib, kb);
                        load_vrows(ib, vb);
                        logits(ch, ka, s);
                        output(ch, s, va);
                        __builtin_amdgcn_sched_barrier(0);
                        ib = load_idx(ch + 3);
                        load_krows(ia, ka);
                        load_vrows(ia, va);
                        logits(ch + 1, kb, s);
                        output(ch + 1, s, vb);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        }
        if constexpr (PM == kPModeRowScaled) {
#pragma unroll
            for (int j = 0; j < HC; ++j) {
                l[j] = row16_sum(l[j]);
                inv_l[j] = l[j] > 0.f ? 1.0f / l[j] : 0.f;
            }
        }
        if constexpr (VB == 4) {
            // tile row c's sum of P over all slots (the four lane groups hold
            // a quarter of every chunk each), then 8 * sum(P) of tile row
            // 4g + j off its accumulators
            int s = psum;
            s += lane_read(s, lane ^ 16);
            s += lane_read(s, lane ^ 32);
#pragma unroll
            for (int i = 0; i < HC; ++i) {
                const u32 corr = 8u * (u32)lane_read(s, 4 * g + i);
#pragma unroll
                for (int b = 0; b < 4; ++b) oacc[b][i] = (int)((u32)oacc[b][i] - corr);
            }
        }
        // rows row0 + i, columns 4c + b
        if (chome) {
#pragma unroll
            for (int i = 0; i < HC; ++i) {
                const size_t orow = (size_t)(i_row * V + row0 + i) * kHeadDim + 4 * c;
                if (DBG && M.o_int)
                    *reinterpret_cast<v4i *>(M.o_int + orow) = v4i{oacc[0][i], oacc[1][i], oacc[2][i], oacc[3][i]};
                // same float operations as dequant_kernel with/without a row scale
                const float rs = PM == kPModeRowScaled ? inv_l[i] : 1.f;
                float4 of;
                of.x = ((float)oacc[0][i] * M.o_scale) * rs;
                of.y = ((float)oacc[1][i] * M.o_scale) * rs;
                of.z = ((float)oacc[2][i] * M.o_scale) * rs;
                of.w = ((float)oacc[3][i] * M.o_scale) * rs;
                if (M.o16) {
                    // fp16 (round to nearest even) straight into a strided
                    // [L][row stride] layout, e.g. the [L][batch][heads * 64]
                    // input of the output projection
                    const __half2 h01 = __floats2half2_rn(of.x, of.y), h23 = __floats2half2_rn(of.z, of.w);
                    const size_t hrow = (size_t)(i_row * V + row0 + i) * (size_t)M.o16_stride + 4 * c;
                    *reinterpret_cast<v2i *>(M.o16 + hrow) =
                        v2i{*reinterpret_cast<const int *>(&h01), *reinterpret_cast<const int *>(&h23)};
                } else {
                    *reinterpret_cast<float4 *>(M.o + orow) = of;
                }
            }
        }
    }
}

}  // namespace mc

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
namespace {

inline unsigned grid_for(long long work, long long per_block) {
    long long b = (work + per_block - 1) / per_block;
    if (b < 1) b = 1;
    if (b > 65535) b = 65535;
    return (unsigned)b;
}

}  // namespace

extern "C" {

mc_status mc_attn_quantize_batched(const mc_quant_job *jobs, int njobs, int bits, int rounding,
                                   long long max_count, hipStream_t stream) {
    if (bits != 8 && bits != 4) return MC_EUNSUPPORTED;
    if ((rounding & ~MC_QUANT_RANGE4) != MC_ROUND_TRUNC && (rounding & ~MC_QUANT_RANGE4) != MC_ROUND_NEAREST)
        return MC_EINVAL_ARG;
    if (njobs < 0 || max_count < 0) return MC_EINVAL_ARG;
    if (njobs == 0 || max_count == 0) return MC_OK;
    if (!jobs || njobs > 65535) return MC_EINVAL_ARG;
    const unsigned gx = grid_for((max_count + 7) / 8, 256 * mc::kQuantGroups);
    const auto *dj = reinterpret_cast<const mc::QuantJob *>(jobs);
    if (bits == 8) hipLaunchKernelGGL(mc::quantize_kernel<8>, dim3(gx, njobs), dim3(256), 0, stream, dj, rounding);
    else hipLaunchKernelGGL(mc::quantize_kernel<4>, dim3(gx, njobs), dim3(256), 0, stream, dj, rounding);
    return mc::check_launch();
}

mc_status mc_attn_quantize(const void *x_fp16, long long count, float scale, int bits, int rounding, void *out,
                           hipStream_t stream) {
    if (bits != 8 && bits != 4) return MC_EUNSUPPORTED;
    if ((rounding & ~MC_QUANT_RANGE4) != MC_ROUND_TRUNC && (rounding & ~MC_QUANT_RANGE4) != MC_ROUND_NEAREST)
        return MC_EINVAL_ARG;
    if (count < 0) return MC_EINVAL_ARG;
    if (count == 0) return MC_OK;
    if (!x_fp16 || !out) return MC_EINVAL_ARG;
    const unsigned gx = grid_for((count + 7) / 8, 256 * mc::kQuantGroups);
    const mc::QuantJob job{static_cast<const __half *>(x_fp16), count, scale, out, 0, 0};
    if (bits == 8) hipLaunchKernelGGL(mc::quantize_one_kernel<8>, dim3(gx), dim3(256), 0, stream, job, rounding);
    else hipLaunchKernelGGL(mc::quantize_one_kernel<4>, dim3(gx), dim3(256), 0, stream, job, rounding);
    return mc::check_launch();
}

mc_status mc_attn_absmax(const void *x_fp16, long long count, unsigned *out_bits, hipStream_t stream) {
    if (count < 0 || !out_bits) return MC_EINVAL_ARG;
    if (count == 0) return MC_OK;
    if (!x_fp16) return MC_EINVAL_ARG;
    hipLaunchKernelGGL(mc::absmax_kernel, dim3(grid_for(count, 256 * 16)), dim3(256), 0, stream,
                       static_cast<const __half *>(x_fp16), count, out_bits);
    return mc::check_launch();
}

mc_status mc_attn_dequant(const int *in, int rows, int cols, float scale, const float *row_scale, float *out,
                          hipStream_t stream) {
    if (rows < 0 || cols <= 0) return MC_EINVAL_SHAPE;
    const long long count = (long long)rows * cols;
    if (count == 0) return MC_OK;
    if (!in || !out) return MC_EINVAL_ARG;
    hipLaunchKernelGGL(mc::dequant_kernel, dim3(grid_for(count, 256 * 8)), dim3(256), 0, stream, in, count, cols,
                       scale, row_scale, out);
    return mc::check_launch();
}

mc_status mc_attn_dequant_f16(const int *in, long long count, float divisor, void *out_f16, hipStream_t stream) {
    if (count < 0) return MC_EINVAL_SHAPE;
    if (count == 0) return MC_OK;
    if (!in || !out_f16) return MC_EINVAL_ARG;
    hipLaunchKernelGGL(mc::dequant_f16_kernel, dim3(grid_for(count, 256 * 8)), dim3(256), 0, stream, in, count,
                       divisor, static_cast<__half *>(out_f16));
    return mc::check_launch();
}

mc_status mc_attn_softmax_f16(int batch, int rows, int vec_length, const int *row_indices, const int *row_offsets,
                              const void *values_f16, long long values_stride, float sqrt_dk, float scale, int bits,
                              void *attn, long long attn_stride_bytes, hipStream_t stream) {
    if (bits != 16 && bits != 8 && bits != 4) return MC_EUNSUPPORTED;
    if (!mc::valid_v(vec_length)) return MC_EINVAL_V;
    if (rows < 0 || batch < 1 || batch > 65535 || values_stride < 0 || attn_stride_bytes < 0) return MC_EINVAL_SHAPE;
    if (rows == 0) return MC_OK;
    if (!row_offsets || !values_f16 || !attn) return MC_EINVAL_ARG;
    // 16-byte loads of the eight fp16 logits of a slot
    if (vec_length == 8 && ((reinterpret_cast<uintptr_t>(values_f16) & 15u) != 0 || values_stride % 8 != 0))
        return MC_EINVAL_ARG;
    constexpr int WPB = 4;
    const dim3 grid((unsigned)((rows + WPB - 1) / WPB), (unsigned)batch), block(64 * WPB);
    const auto *vals = static_cast<const __half *>(values_f16);
    auto *out = static_cast<unsigned char *>(attn);
#define MC_REF_SOFTMAX(V_, B_)                                                                                     \
    hipLaunchKernelGGL((mc::ref_softmax_kernel<V_, B_, WPB>), grid, block, 0, stream, rows, row_indices,           \
                       row_offsets, vals, values_stride, sqrt_dk, scale, out, attn_stride_bytes)
#define MC_REF_SOFTMAX_V(B_)                                                                                       \
    switch (vec_length) {                                                                                          \
    case 2: MC_REF_SOFTMAX(2, B_); break;                                                                          \
    case 4: MC_REF_SOFTMAX(4, B_); break;                                                                          \
    default: MC_REF_SOFTMAX(8, B_); break;                                                                         \
    }
    if (bits == 16) { MC_REF_SOFTMAX_V(16) }
    else if (bits == 8) { MC_REF_SOFTMAX_V(8) }
    else { MC_REF_SOFTMAX_V(4) }
#undef MC_REF_SOFTMAX_V
#undef MC_REF_SOFTMAX
    return mc::check_launch();
}

mc_status mc_attn_zero_gaps(int batch, int rows, const int *row_offsets, int slots, int group, int slot_bits, void *out,
                            long long stride_bytes, hipStream_t stream) {
    if (batch < 1 || batch > 65535 || rows < 0 || slots < 0 || stride_bytes < 0) return MC_EINVAL_SHAPE;
    if (group < 1 || slot_bits < 8 || slot_bits % 8 != 0) return MC_EINVAL_ARG;
    if (slots == 0) return MC_OK;
    if (!out || (rows > 0 && !row_offsets)) return MC_EINVAL_ARG;
    return mc::zero_gaps(batch, rows, row_offsets, slots, group, slot_bits, out, stride_bytes, stream);
}

mc_status mc_attn_softmax_requant(int m_vec, int vec_length, const int *row_indices, const int *row_offsets,
                                  const int *s_vals, float alpha, float p_scale, int p_mode, void *p_out,
                                  float *row_inv_l, hipStream_t stream) {
    if (p_mode != MC_P_REFERENCE && p_mode != MC_P_ROW_SCALED && p_mode != MC_P_REFERENCE_4BIT) return MC_EINVAL_ARG;
    if (!mc::valid_v(vec_length)) return MC_EINVAL_V;
    if (m_vec < 0) return MC_EINVAL_SHAPE;
    if (m_vec == 0) return MC_OK;
    if (!row_offsets || !s_vals || !p_out) return MC_EINVAL_ARG;
    constexpr int WPB = 4;
    const dim3 grid((m_vec + WPB - 1) / WPB), block(64 * WPB);
    auto *po = static_cast<unsigned char *>(p_out);
    switch (vec_length) {
    case 2: hipLaunchKernelGGL((mc::softmax_requant_kernel<2, WPB>), grid, block, 0, stream, m_vec, row_indices, row_offsets, s_vals, alpha, p_scale, p_mode, po, row_inv_l); break;
    case 4: hipLaunchKernelGGL((mc::softmax_requant_kernel<4, WPB>), grid, block, 0, stream, m_vec, row_indices, row_offsets, s_vals, alpha, p_scale, p_mode, po, row_inv_l); break;
    default: hipLaunchKernelGGL((mc::softmax_requant_kernel<8, WPB>), grid, block, 0, stream, m_vec, row_indices, row_offsets, s_vals, alpha, p_scale, p_mode, po, row_inv_l); break;
    }
    return mc::check_launch();
}

mc_status mc_attn_forward(const mc_attn_matrix *matrices, const int *items, int n_items, int qk_bits, int v_bits,
                          int vec_length, float p_scale, int p_mode, int grid_waves, int debug, hipStream_t stream) {
    if (qk_bits != 8 && qk_bits != 4) return MC_EUNSUPPORTED;
    if (v_bits != 8 && !(v_bits == 4 && qk_bits == 4)) return MC_EUNSUPPORTED;
    if (p_mode != MC_P_REFERENCE && p_mode != MC_P_ROW_SCALED && p_mode != MC_P_REFERENCE_4BIT) return MC_EINVAL_ARG;
    if (!mc::valid_v(vec_length)) return MC_EINVAL_V;
    if (n_items < 0 || grid_waves < 0) return MC_EINVAL_ARG;
    if (n_items == 0) return MC_OK;
    if (!matrices || !items) return MC_EINVAL_ARG;
    constexpr int WPB = 4;
    long long waves = grid_waves > 0 ? grid_waves : n_items;
    if (waves > n_items) waves = n_items;
    const dim3 grid((unsigned)((waves + WPB - 1) / WPB)), block(64 * WPB);
    const auto *mats = reinterpret_cast<const mc::AttnMatrix *>(matrices);
    const auto *its = reinterpret_cast<const int2 *>(items);
#define MC_ATTN_LAUNCH(V_, B_, VB_, PM_)                                                                             \
    do {                                                                                                             \
        if (debug)                                                                                                   \
            hipLaunchKernelGGL((mc::attention_kernel<V_, B_, VB_, PM_, WPB, true>), grid, block, 0, stream, mats,    \
                               its, n_items, p_scale);                                                               \
        else                                                                                                         \
            hipLaunchKernelGGL((mc::attention_kernel<V_, B_, VB_, PM_, WPB, false>), grid, block, 0, stream, mats,   \
                               its, n_items, p_scale);                                                               \
    } while (0)
#define MC_ATTN_LAUNCH_P(V_, B_, VB_)                                                                                \
    switch (p_mode) {                                                                                                \
    case MC_P_REFERENCE: MC_ATTN_LAUNCH(V_, B_, VB_, 0); break;                                                      \
    case MC_P_ROW_SCALED: MC_ATTN_LAUNCH(V_, B_, VB_, 1); break;                                                     \
    default: MC_ATTN_LAUNCH(V_, B_, VB_, 2); break;                                                                  \
    }
#define MC_ATTN_LAUNCH_V(B_, VB_)                                                                                    \
    switch (vec_length) {                                                                                            \
    case 2: MC_ATTN_LAUNCH_P(2, B_, VB_); break;                                                                     \
    case 4: MC_ATTN_LAUNCH_P(4, B_, VB_); break;                                                                     \
    default: MC_ATTN_LAUNCH_P(8, B_, VB_); break;                                                                    \
    }
    if (qk_bits == 8) { MC_ATTN_LAUNCH_V(8, 8) }
    else if (v_bits == 8) { MC_ATTN_LAUNCH_V(4, 8) }
    else { MC_ATTN_LAUNCH_V(4, 4) }
#undef MC_ATTN_LAUNCH_P
#undef MC_ATTN_LAUNCH_V
#undef MC_ATTN_LAUNCH
    return mc::check_launch();
}

}  // extern "C"
