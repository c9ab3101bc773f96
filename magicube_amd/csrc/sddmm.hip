// C ABI of the SDDMM family: validation and dispatch.
#include "mc_internal.hpp"
#include "sddmm_kernel.hpp"

namespace mc {
namespace {

constexpr int kMaxWaves = 8;   // waves per row

// Waves per row W and tiles per group T.  Under 768 rows (times the batch) a
// launch is one round of workgroups, so a row is spread over more waves and,
// at K <= 128, single tiles; from there on fewer waves with longer pipelines
// keep more rows resident (819 rows x 5463, K = 448, 93 % sparse, operands not
// in the caches: W4 18.9 us, W8 23.3).  At K = 256 two tiles' gathers take the
// registers of a wave more per SIMD: T1 (1000 rows x 8000, 80 % sparse: 28.2
// against 30.5 us; 819 rows, K = 192: 10.9 against 12.3).  Measured on MI355X, us (rows x N, K, sparsity):
//                            W8 T1   W8 T2   W4 T1   W4 T2   W2 T2   W16 T1
//   512 x 4096, 64, 0.9        4.9     5.0     5.7     5.6     7.3     5.6
//   512 x 4096, 128, 0.9       5.4     5.6     6.1     6.1     7.8     6.6
//   256 x 2304, 512, 0.9       5.8     5.3     6.2     6.0     7.0     (8 at most)
//   1024 x 8192, 64, 0.9      11.6    11.1    11.2    10.6    13.2    13.0
//   1024 x 8192, 128, 0.9     13.5    12.8    12.8    12.4    14.7    15.5
//   1024 x 8192, 512, 0.9     35.9    28.6    30.9    26.7    28.7
// against 5.1, 7.0, 7.7, 11.7, 18.7 and 54.3 for 16 (K = 64) or 8 waves with
// gathers in the operand layout and nothing in flight across groups.  16-bit
// operands (two digits) keep one tile: 10.8 against 11.3 at K = 512.
template <int V, int BITS, bool SGN, int NKC, int TPW, int OUT>
mc_status sddmm_launch_tiles(const SddmmArgs &a, int waves, int batch, hipStream_t s) {
    hipLaunchKernelGGL((sddmm_kernel<V, BITS, SGN, NKC, TPW, kMaxWaves, OUT>), dim3((unsigned)a.m_vec, (unsigned)batch),
                       dim3(64 * waves), 0, s, a);
    return check_launch();
}

template <int V, int BITS, bool SGN, int NKC, int OUT>
mc_status sddmm_launch(const SddmmArgs &a, int batch, hipStream_t s) {
    const bool one_round = (long long)a.m_vec * batch < 768;
    const int waves = one_round ? 8 : 4;
    if constexpr (BITS == 16 || NKC == 4) {
        return sddmm_launch_tiles<V, BITS, SGN, NKC, 1, OUT>(a, waves, batch, s);
    } else {
        if constexpr (NKC <= 2) {
            if (one_round) return sddmm_launch_tiles<V, BITS, SGN, NKC, 1, OUT>(a, waves, batch, s);
        }
        return sddmm_launch_tiles<V, BITS, SGN, NKC, 2, OUT>(a, waves, batch, s);
    }
}

template <int V, int BITS, bool SGN, int OUT>
mc_status sddmm_launch_k(int nkc, const SddmmArgs &a, int batch, hipStream_t s) {
    switch (nkc) {
    case 1: return sddmm_launch<V, BITS, SGN, 1, OUT>(a, batch, s);
    case 2: return sddmm_launch<V, BITS, SGN, 2, OUT>(a, batch, s);
    case 4: return sddmm_launch<V, BITS, SGN, 4, OUT>(a, batch, s);
    case 8: return sddmm_launch<V, BITS, SGN, 8, OUT>(a, batch, s);
    default: return MC_EUNSUPPORTED;
    }
}

template <int BITS, bool SGN, int OUT>
mc_status sddmm_launch_v(int V, int nkc, const SddmmArgs &a, int batch, hipStream_t s) {
    switch (V) {
    case 2: return sddmm_launch_k<2, BITS, SGN, OUT>(nkc, a, batch, s);
    case 4: return sddmm_launch_k<4, BITS, SGN, OUT>(nkc, a, batch, s);
    case 8: return sddmm_launch_k<8, BITS, SGN, OUT>(nkc, a, batch, s);
    default: return MC_EINVAL_V;
    }
}

template <int BITS>
mc_status sddmm_launch_all(bool sgn, bool ref, int V, int nkc, const SddmmArgs &a, int batch, hipStream_t s) {
    if (sgn)
        return ref ? sddmm_launch_v<BITS, true, kOutReference>(V, nkc, a, batch, s)
                   : sddmm_launch_v<BITS, true, kOutVector>(V, nkc, a, batch, s);
    return ref ? sddmm_launch_v<BITS, false, kOutReference>(V, nkc, a, batch, s)
               : sddmm_launch_v<BITS, false, kOutVector>(V, nkc, a, batch, s);
}

mc_status sddmm_entry(int bits, mc_signedness sign, int layout, int m_vec, int k, int n, const int *row_indices,
                      const int *row_offsets, const int *col_indices, const int *lhs_matrix, const int *rhs_matrix,
                      int *output_values, int vec_length, hipStream_t stream, int batch = 1,
                      long long lhs_stride = 0, long long rhs_stride = 0, long long out_stride = 0,
                      __half *out16 = nullptr, float divisor = 1.f, int slots = 0) {
    if (batch < 1 || batch > 65535 || lhs_stride < 0 || rhs_stride < 0 || out_stride < 0) return MC_EINVAL_SHAPE;
    if ((lhs_stride | rhs_stride) & 3) return MC_EINVAL_SHAPE;   // every matrix starts dword aligned
    if (bits != 16 && bits != 8 && bits != 4) return MC_EUNSUPPORTED;
    if (sign != MC_SIGNED && sign != MC_UNSIGNED) return MC_EINVAL_ARG;
    if (layout != MC_SDDMM_OUT_REFERENCE && layout != MC_SDDMM_OUT_VECTOR) return MC_EINVAL_ARG;
    if (!valid_v(vec_length)) return MC_EINVAL_V;
    if (m_vec < 0 || n <= 0 || k <= 0 || k % 64 != 0) return MC_EINVAL_SHAPE;
    // 64-deep chunks held per pass: the smallest of 1, 2, 4, 8 that covers k,
    // else 8 with several passes
    const int chunks = k / 64;
    const int nkc = chunks <= 1 ? 1 : chunks <= 2 ? 2 : chunks <= 4 ? 4 : 8;
    const long long lhs_bytes = (long long)m_vec * vec_length * k * bits / 8;
    const long long rhs_bytes = (long long)n * k * bits / 8;
    if (lhs_bytes >= (1LL << 30) || rhs_bytes >= (1LL << 30)) return MC_EINVAL_SHAPE;
    if (m_vec == 0) return MC_OK;
    if (!row_offsets || !col_indices || !lhs_matrix || !rhs_matrix || !(output_values || out16)) return MC_EINVAL_ARG;
    SddmmArgs a{};
    a.m_vec = m_vec;
    a.k = k;
    a.n = n;
    a.row_indices = row_indices;
    a.row_offsets = row_offsets;
    a.col_indices = col_indices;
    a.lhs = reinterpret_cast<const unsigned char *>(lhs_matrix);
    a.rhs = reinterpret_cast<const unsigned char *>(rhs_matrix);
    a.out = output_values;
    a.lhs_bytes = (unsigned)lhs_bytes;
    a.rhs_bytes = (unsigned)rhs_bytes;
    a.lhs_stride = lhs_stride;
    a.rhs_stride = rhs_stride;
    a.out_stride = out_stride;
    if (out16) {
        if (k > 512 || bits == 16) return MC_EUNSUPPORTED;   // one pass over K
        // a lane's rows of a slot are stored together: 8 bytes, 4 at V = 2
        const long long unit = vec_length == 2 ? 4 : 8;
        if ((reinterpret_cast<uintptr_t>(out16) | (unsigned long long)(batch > 1 ? 2 * out_stride : 0)) & (unit - 1))
            return MC_EINVAL_ARG;
        a.out16 = out16;
        a.div = make_divisor(divisor);
        if (a.div.y == 0.f) return MC_EUNSUPPORTED;
        const mc_status st = zero_gaps(batch, m_vec, row_offsets, slots, 8, 16 * vec_length, out16, 2 * out_stride,
                                       stream);
        if (st != MC_OK) return st;
        return bits == 8 ? sddmm_launch_v<8, true, kOutHalf>(vec_length, nkc, a, batch, stream)
                         : sddmm_launch_v<4, true, kOutHalf>(vec_length, nkc, a, batch, stream);
    }
    const bool sgn = sign == MC_SIGNED, ref = layout == MC_SDDMM_OUT_REFERENCE;
    if (bits == 16) return sddmm_launch_all<16>(sgn, ref, vec_length, nkc, a, batch, stream);
    return bits == 8 ? sddmm_launch_all<8>(sgn, ref, vec_length, nkc, a, batch, stream)
                     : sddmm_launch_all<4>(sgn, ref, vec_length, nkc, a, batch, stream);
}

}  // namespace
}  // namespace mc

extern "C" {

mc_status mc_sddmm_l8r8(int m_vec, int k, int n, const int *row_indices, const int *row_offsets,
                        const int *col_indices, const int *lhs_matrix, const int *rhs_matrix, int *output_values,
                        int vec_length, mc_signedness sign, hipStream_t stream) {
    return mc::sddmm_entry(8, sign, MC_SDDMM_OUT_REFERENCE, m_vec, k, n, row_indices, row_offsets, col_indices,
                           lhs_matrix, rhs_matrix, output_values, vec_length, stream);
}

mc_status mc_sddmm_l4r4(int m_vec, int k, int n, const int *row_indices, const int *row_offsets,
                        const int *col_indices, const int *lhs_matrix, const int *rhs_matrix, int *output_values,
                        int vec_length, mc_signedness sign, hipStream_t stream) {
    return mc::sddmm_entry(4, sign, MC_SDDMM_OUT_REFERENCE, m_vec, k, n, row_indices, row_offsets, col_indices,
                           lhs_matrix, rhs_matrix, output_values, vec_length, stream);
}

mc_status mc_sddmm_l16r16(int m_vec, int k, int n, const int *row_indices, const int *row_offsets,
                          const int *col_indices, const int *lhs_matrix, const int *rhs_matrix, int *output_values,
                          int vec_length, mc_signedness sign, hipStream_t stream) {
    return mc::sddmm_entry(16, sign, MC_SDDMM_OUT_REFERENCE, m_vec, k, n, row_indices, row_offsets, col_indices,
                           lhs_matrix, rhs_matrix, output_values, vec_length, stream);
}

mc_status mc_sddmm_run(int bits, mc_signedness sign, int layout, int m_vec, int k, int n, const int *row_indices,
                       const int *row_offsets, const int *col_indices, const int *lhs_matrix,
                       const int *rhs_matrix, int *output_values, int vec_length, hipStream_t stream) {
    return mc::sddmm_entry(bits, sign, layout, m_vec, k, n, row_indices, row_offsets, col_indices, lhs_matrix,
                           rhs_matrix, output_values, vec_length, stream);
}

mc_status mc_sddmm_batched(int bits, mc_signedness sign, int layout, int batch, int m_vec, int k, int n,
                           const int *row_indices, const int *row_offsets, const int *col_indices,
                           const int *lhs_matrix, long long lhs_stride_bytes, const int *rhs_matrix,
                           long long rhs_stride_bytes, int *output_values, long long out_stride, int vec_length,
                           hipStream_t stream) {
    return mc::sddmm_entry(bits, sign, layout, m_vec, k, n, row_indices, row_offsets, col_indices, lhs_matrix,
                           rhs_matrix, output_values, vec_length, stream, batch, lhs_stride_bytes,
                           rhs_stride_bytes, out_stride);
}

mc_status mc_sddmm_batched_f16(int bits, int batch, int m_vec, int k, int n, const int *row_indices,
                               const int *row_offsets, const int *col_indices, int slots, const int *lhs_matrix,
                               long long lhs_stride_bytes, const int *rhs_matrix, long long rhs_stride_bytes,
                               float divisor, void *out_f16, long long out_stride, int vec_length,
                               hipStream_t stream) {
    if (slots < 0) return MC_EINVAL_SHAPE;
    if (m_vec > 0 && !out_f16) return MC_EINVAL_ARG;
    return mc::sddmm_entry(bits, MC_SIGNED, MC_SDDMM_OUT_VECTOR, m_vec, k, n, row_indices, row_offsets, col_indices,
                           lhs_matrix, rhs_matrix, nullptr, vec_length, stream, batch, lhs_stride_bytes,
                           rhs_stride_bytes, out_stride, static_cast<__half *>(out_f16), divisor, slots);
}

}  // extern "C"
