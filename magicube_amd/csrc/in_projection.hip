// The attention module's in-projection y = half(x w^T + bias) on many rows,
// accumulated in fp32, which quantizes K and V as it stores them.  The
// reference leaves the product to torch and quantizes in a launch of its own
// (end2end_eval/sparse_transformer_magicube/spattention.py).
#include <hip/hip_fp16.h>

#include "attention_common.hpp"
#include "mc_internal.hpp"

namespace mc {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));

constexpr int kTileM = 128, kTileN = 128, kTileK = 64;     // rows of x, columns of y, depth of one stage
constexpr int kMaxCols = 4096, kMaxMats = 256;             // bias columns and (sample, head) matrices held in LDS
constexpr int kWave = 64;                                  // a wave's tile: 64 rows x 64 columns

struct ProjectionArgs {
    long long rows;
    int n, k;
    const __half *x;            // [rows][k]
    const __half *w;            // [n][k]
    const __half *bias;         // [n] or null
    __half *out;                // [rows][n]: its Q columns
    // row l * samples + b, columns [Q | K | V] of heads x 64
    const AttnMatrix *mats;     // matrix b * heads + h
    int samples, heads;
    float scale;
    int v_range4;
};

__device__ __forceinline__ v4f mfma_f16(const v4i &a, const v4i &b, const v4f &c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const half8 *>(&a),
                                                  *reinterpret_cast<const half8 *>(&b), c, 0, 0, 0);
}
__device__ __forceinline__ __half2 as_half2(int x) { return *reinterpret_cast<const __half2 *>(&x); }
__device__ __forceinline__ int as_int(const __half2 &x) { return *reinterpret_cast<const int *>(&x); }

// KB: bits per K value.
//
// y^T = w x^T on the matrix cores, so that a lane's accumulators are 16
// consecutive columns of one row: the rows of w go to LDS in the order that
// makes them so, a row leaves as 128 contiguous bytes per four lanes, and a
// head's 64 quantized columns as one 64-byte line.  Both operands pass
// through LDS in 64-deep stages of 128-byte rows, whose 16-byte pieces are
// xor-ed with the row (no bank conflicts for the writes or the MFMA reads).
// Persistent workgroups, two per CU, walk (row block, column block) tiles:
// the next stage's loads, of the next tile at a tile's end, are in flight
// while a stage is multiplied or a tile stored.  An XCD takes whole row
// blocks, so that x crosses HBM once and the column blocks read it from L2.
//
// 32768 rows of 256 to 768 take 30 us in a kernel trace and 27 in a row, where
// torch's product takes 27 and a quantize launch of K and V 10 to 12 (one after
// the other 40); a batch-8 attention module of L = 4096, E = 256 went from 126.6
// to 107.0 us.  There TD is busy 44 % of the time (57 % of it waiting), TA 31,
// VALU 24, LDS 16 without bank conflicts, MFMA 15: bound by the latency of its
// stages.  At that size one and a half workgroups per CU take 33-35 us and one
// tile per workgroup 28-30 against 27-28.  By passes of the module, two stages'
// loads kept in flight over the barrier, the next stage written to LDS under
// the products, three workgroups per CU with 32-deep stages and 256-row tiles
// were 0-2 % slower.
template <int KB>
__global__ __launch_bounds__(256, 2) void in_projection_kernel(ProjectionArgs a, int mb, int nb) {
    __shared__ v4i xs[2][kTileM * 8], ws[2][kTileN * 8];
    // bias and K / V buffers: from LDS, because a wait for a load at a tile's
    // end would also wait for the stages under way
    __shared__ __attribute__((aligned(16))) __half bs[kMaxCols];
    __shared__ unsigned char *kv[2][kMaxMats];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int wm = (wave & 1) * kWave, wn = (wave >> 1) * kWave;
    const int xcd = blockIdx.x & 7, step = gridDim.x >> 3;
    const int tiles = xcd < mb ? ((mb - xcd + 7) >> 3) * nb : 0;
    const int nk = a.k / kTileK;

    // staging: thread t moves piece t % 8 of rows t / 8 + 32 i
    const int piece = tid & 7, srow = tid >> 3;
    const int sslot = srow * 8 + (piece ^ (srow & 7));        // + 256 i: the row's low bits do not change
    struct Stage {
        v4i x[4], w[4];
    };
    int next_tile = blockIdx.x >> 3, next_kc = 0;                // the next stage to load
    u32 wrow[4];                                                 // LDS row 16 j + c of a wave's 64 is
#pragma unroll                                                   // column 16 (c / 4) + 4 j + c % 4
    for (int i = 0; i < 4; ++i) {
        const int r = srow + 32 * i;
        const int col = (r & 64) + 16 * ((r >> 2) & 3) + 4 * ((r >> 4) & 3) + (r & 3);
        wrow[i] = (u32)(col * a.k + piece * 8) * 2u;
    }
    // past the walk's end the last stage is loaded again (and not used)
    const auto load = [&](Stage &s) {
        const int rb = next_tile / nb;
        const long long m0 = (long long)(xcd + 8 * rb) * kTileM;
        const int n0 = (next_tile - rb * nb) * kTileN;
        const int top = (int)min(a.rows - 1 - m0, (long long)kTileM);   // rows past the end repeat the last, and are not stored
        const char *xb = reinterpret_cast<const char *>(a.x + m0 * a.k + next_kc * kTileK);
        const char *wb = reinterpret_cast<const char *>(a.w + (long long)n0 * a.k + next_kc * kTileK);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const u32 xo = (u32)(min(srow + 32 * i, top) * a.k + piece * 8) * 2u;
            s.x[i] = *reinterpret_cast<const v4i *>(xb + xo);
            s.w[i] = *reinterpret_cast<const v4i *>(wb + wrow[i]);
        }
        const int kc1 = next_kc + 1 == nk ? 0 : next_kc + 1, tile1 = next_tile + (kc1 ? 0 : step);
        if (tile1 < tiles) {
            next_kc = kc1;
            next_tile = tile1;
        }
    };
    const auto stage = [&](const Stage &s, int buf) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            xs[buf][sslot + 256 * i] = s.x[i];
            ws[buf][sslot + 256 * i] = s.w[i];
        }
    };

    int tile = next_tile, kc = 0;                                // the stage being multiplied
    if (tile >= tiles) return;                                   // the whole workgroup
    v4f acc[4][4];                                               // [row tile][column quad j]
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[m][j] = v4f{0.f, 0.f, 0.f, 0.f};
    Stage ra, rb;                                                // stages it + 1 and it + 2 of the walk
    for (int i = tid; i < a.n; i += 256) bs[i] = a.bias ? a.bias[i] : __half(0.f);
    for (int i = tid; i < a.samples * a.heads; i += 256) {
        kv[0][i] = const_cast<unsigned char *>(a.mats[i].k);
        kv[1][i] = const_cast<unsigned char *>(a.mats[i].v);
    }
    load(ra);
    __builtin_amdgcn_sched_barrier(0);
    load(rb);
    __builtin_amdgcn_sched_barrier(0);
    stage(ra, 0);
    load(ra);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    // one stage from LDS buffer `buf`; s holds the next one
    const auto body = [&](Stage &s, int buf) {
        const bool last = kc == nk - 1;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            v4i xf[4], wf[4];
            const int p = (g + 4 * ks) ^ (c & 7);
#pragma unroll
            for (int m = 0; m < 4; ++m) xf[m] = xs[buf][(wm + 16 * m + c) * 8 + p];
#pragma unroll
            for (int j = 0; j < 4; ++j) wf[j] = ws[buf][(wn + 16 * j + c) * 8 + p];
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[m][j] = mfma_f16(wf[j], xf[m], acc[m][j]);
        }
        if (last) {
            const long long m0 = (long long)(xcd + 8 * (tile / nb)) * kTileM + wm;
            const int n0 = tile % nb * kTileN + wn;              // wave-uniform: one head's columns
            const v4i b0 = *reinterpret_cast<const v4i *>(bs + n0 + 16 * g),
                      b1 = *reinterpret_cast<const v4i *>(bs + n0 + 16 * g + 8);
            const int head = n0 >> 6, part = head / a.heads;
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const long long row = m0 + 16 * m + c;
                __half2 y[8];                                    // columns n0 + 16 g ..., as the layer stores them
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const __half2 b = as_half2(e < 4 ? b0[e & 3] : b1[e & 3]);
                    y[e] = __floats2half2_rn(acc[m][e >> 1][2 * (e & 1)] + __low2float(b),
                                             acc[m][e >> 1][2 * (e & 1) + 1] + __high2float(b));
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[m][j] = v4f{0.f, 0.f, 0.f, 0.f};
                if (row >= a.rows) continue;
                if (part == 0) {
                    const size_t o = (size_t)row * a.n + n0 + 16 * g;
                    *reinterpret_cast<v4i *>(a.out + o) = v4i{as_int(y[0]), as_int(y[1]), as_int(y[2]), as_int(y[3])};
                    *reinterpret_cast<v4i *>(a.out + o + 8) = v4i{as_int(y[4]), as_int(y[5]), as_int(y[6]), as_int(y[7])};
                } else {
                    // the quantize launch's expression (quantize_group), truncating
                    const bool range4 = part == 1 ? KB == 4 : a.v_range4 != 0;
                    const float lo = range4 ? -8.f : -128.f, hi = range4 ? 7.f : 127.f;
                    u32 q[16];
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const float f = (e & 1 ? __high2float(y[e >> 1]) : __low2float(y[e >> 1])) * a.scale;
                        q[e] = (u32)(int)fminf(fmaxf(f, lo), hi);
                    }
                    const int r32 = (int)row, l = r32 / a.samples, b = r32 - l * a.samples;
                    unsigned char *o = kv[part - 1][b * a.heads + head - part * a.heads];
                    if (KB == 4 && part == 1) {
                        u32 t[2] = {0, 0};
#pragma unroll
                        for (int e = 0; e < 16; ++e) t[e >> 3] |= (q[e] & 15u) << (4 * (e & 7));
                        *reinterpret_cast<v2i *>(o + (size_t)l * 32 + 8 * g) = v2i{(int)t[0], (int)t[1]};
                    } else {
                        v4i t;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            t[e] = (int)((q[4 * e] & 255) | (q[4 * e + 1] & 255) << 8 | (q[4 * e + 2] & 255) << 16 |
                                         q[4 * e + 3] << 24);
                        *reinterpret_cast<v4i *>(o + (size_t)l * 64 + 16 * g) = t;
                    }
                }
            }
        }
        kc = last ? 0 : kc + 1;
        tile += last ? step : 0;
        if (tile >= tiles) return false;
        stage(s, buf ^ 1);
        load(s);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        return true;
    };
    while (body(rb, 0) && body(ra, 1)) {
    }
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

template <int KB> mc_status in_projection_launch(const ProjectionArgs &a, hipStream_t stream) {
    const int mb = (int)((a.rows + kTileM - 1) / kTileM), nb = a.n / kTileN;
    const long long per_xcd = (long long)((mb + 7) / 8) * nb;
    if (per_xcd > 0x3FFFFFFF) return MC_EINVAL_SHAPE;
    const int step = per_xcd < 64 ? (int)per_xcd : 64;           // two workgroups on each of 32 CUs
    hipLaunchKernelGGL((in_projection_kernel<KB>), dim3(8 * step), dim3(256), 0, stream, a, mb, nb);
    return check_launch();
}

}  // namespace
}  // namespace mc

extern "C" {

mc_status mc_attn_in_projection_f16(int seq_len, int samples, int heads, const void *x, const void *w,
                                    const void *bias, float scale, int qk_bits, int v_range4,
                                    const mc_attn_matrix *matrices, void *qkv, hipStream_t stream) {
    if (qk_bits != 8 && qk_bits != 4) return MC_EUNSUPPORTED;
    if (seq_len < 0 || samples <= 0 || heads <= 0 || (long long)samples * heads > mc::kMaxMats) return MC_EINVAL_SHAPE;
    const int e = heads * 64;
    if (e % mc::kTileK || 3 * e % mc::kTileN || 3 * e > mc::kMaxCols || (long long)seq_len * samples >= (1LL << 30))
        return MC_EINVAL_SHAPE;
    if (seq_len == 0) return MC_OK;
    if (!x || !w || !qkv || !matrices) return MC_EINVAL_ARG;
    if (!mc::aligned16(x) || !mc::aligned16(w) || !mc::aligned16(bias) || !mc::aligned16(qkv)) return MC_EINVAL_ARG;
    mc::ProjectionArgs a{};
    a.rows = (long long)seq_len * samples;
    a.n = 3 * e;
    a.k = e;
    a.x = static_cast<const __half *>(x);
    a.w = static_cast<const __half *>(w);
    a.bias = static_cast<const __half *>(bias);
    a.out = static_cast<__half *>(qkv);
    a.mats = reinterpret_cast<const mc::AttnMatrix *>(matrices);
    a.samples = samples;
    a.heads = heads;
    a.scale = scale;
    a.v_range4 = v_range4;
    return qk_bits == 8 ? mc::in_projection_launch<8>(a, stream) : mc::in_projection_launch<4>(a, stream);
}

}  // extern "C"
