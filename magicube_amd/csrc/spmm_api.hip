// C ABI of the SpMM family: argument validation, the tile-config table and
// dispatch to the per-pair instantiation units.  The entry points keep no
// state: the tile is the default for the shape unless the call names one.
#include "spmm_dispatch.hpp"

namespace mc {
namespace {

// MFMA rows of a vector row: its digit planes times its V rows (the planes of
// the pairs in spmm_kernel.hpp).
int mfma_rows(int lhs_bits, int rhs_bits, bool sgn, int V) {
    if (lhs_bits == 4) return V;
    if (lhs_bits == 8) return (sgn ? 1 : 2) * V;
    return (lhs_bits / 4 - (sgn ? 1 : 0)) * V;
}

// Slots per vector row from which wide products take four dwords per lane
// (config 24) instead of one and four waves per row (17).  Short rows do not:
// their gathers cost less than the fewer waves and the store through LDS.
// Measured on MI355X over 5000 shapes (256 to 4096 rows, K 256 to 8192, 2 to 16
// tiles, 16 to 1600 slots, V = 2, 4, 8, every pair of 8- and 16-bit B): by this
// rule 0.5 % above the better of the two on average, always 24 2.8, always 17
// 7.8.  It rests on, us 17 / 24 at 32, 64, 128, 256, 400 slots:
// * the launch: L8-R8, V = 8, K = 1024, 1024 rows, N = 1024 9.3 / 10.0, 10.3 /
//   11.4, 12.7 / 13.5, 20.5 / 20.3, 29.6 / 26.3; N = 4096 26.9 / 26.9, 32.4 /
//   31.8, 41.0 / 40.2, 77.8 / 64.6, 117 / 85; few MFMA rows to recombine (V = 2),
//   N = 2048 13.4 / 12.2, 15.4 / 14.2, 19.1 / 18.3;
// * whole lines: where B's rows start off 64 bytes a wave's 4-byte gathers touch
//   two lines for one, its 16-byte gathers five for four (1024 rows, K = 4096,
//   L8-R8, V = 8, 256 slots: N = 1024 21.0 / 21.0, N = 976 23.7 / 21.6);
// * the XCDs, which workgroups reach in turn: with G workgroups per row (the
//   wide tile has two waves to one, 17 four) an XCD reads 1 / gcd(G, 8) of B.
//   Where the wide tile's XCDs read more than 17's, and more than their L2
//   holds, rows have to be longer (K = 4096, 256, 400, 800 slots: N = 3584 92.9 /
//   111, 134 / 150, 252 / 226; N = 2560 60.4 / 70.7, 87.7 / 90.3, 163 / 127;
//   16-bit B, N = 1792 84.8 / 102, 124 / 138, 241 / 203); where they read as much
//   or less, rows may be shorter (N = 1792, 8-bit, 256 slots 48.5 / 32.7).
int wide_least_slots(int rhs_bits, int n, int k, long long waves, int wide_tiles, int rows) {
    constexpr long long kL2 = 4LL << 20;                        // of one XCD
    const auto parts = [](int g) { return g & 1 ? 1 : g & 2 ? 2 : g & 4 ? 4 : 8; };   // gcd(g, 8)
    const int here = parts((wide_tiles + 1) / 2), narrow = parts(wide_tiles);
    const long long row_bytes = (long long)n * rhs_bits / 8, b_bytes = row_bytes * k;
    const bool lines = row_bytes % 64 == 0;
    const bool more = here < narrow && b_bytes / here > kL2;
    if (more && lines) return 420;
    if (rhs_bits == 16) return 0;                               // faster at every length
    if (more) return 150;
    int least = lines ? 300 : 150;
    if (b_bytes > kL2 && here >= narrow) least = here > narrow ? 50 : least / 2;
    if (rows <= 6 && waves >= (b_bytes <= kL2 ? 4096 : 8192)) return 0;
    if (waves >= 16384) return least < 50 ? least : 50;
    const int full = lines && b_bytes > kL2 ? 160 : 100;
    return waves >= 8192 && full < least ? full : least;
}

// row_slots: slots per vector row on average, 0 where the caller does not know
// (long rows then).
int default_config(int rhs_bits, int n, int k, long long m_vec, int rows, int row_slots) {
    // Four dwords of 8- or 16-bit B per lane where the launch holds 2048 waves
    // of 16 * 4 dwords, two per workgroup (an odd tile's second wave included),
    // and a vector row is one MFMA row tile (two need 128 accumulators and
    // leave two waves per SIMD).  The gathers are bound by L1's address path:
    // a 4-byte load of a wave takes it 8 cycles, a 16-byte one 16.  Measured on
    // MI355X, us, one dword and four waves per row (config 17) against this:
    // L8-R8, V = 8, 8192 x 8192, N = 4096, 90 % sparse 261 / 160; 4096 x 4096,
    // N = 4096, 70 and 90 % 147 / 112, 59 / 45; N = 2048, 90 % 33.5 / 25.6; N =
    // 1024, 70 and 90 % 43 / 32, 16.8 / 14.6; N = 512 (1024 waves) 24.0 / 25.2,
    // 10.1 / 11.7.  L16-R8, V = 4, N = 4096, 80 % 103 / 74; L16-R16, V = 4 252 /
    // 154.  Two row tiles: L16-R8, V = 8 114 / 135, 42 / 62 (config 25: 99, 55).
    // Not for a row of three tiles: the fourth wave has no columns and the
    // third few just past the second, where config 17 fills its waves better
    // (1024 vector rows, K = 4096, 90 %: N = 516 26.0 / 28.5, 580 28.7 / 28.4,
    // 640 22.5 / 25.3, 768 24.0 / 25.9; 512 rows 14.0 / 16.5, 16.1 / 16.9, 13.0
    // / 14.1, 14.3 / 14.4).  Two tiles and four or five are faster from their
    // first column on (1024 rows: 260 20.0 / 13.7, 320 16.3 / 13.4, 772 37.4 /
    // 29.0, 1028 50.8 / 38.6; 512 rows: 772 19.9 / 17.3, 1028 27.9 / 21.7).
    // Nor for rows too short for it (wide_least_slots).
    if (rhs_bits != 4 && rows <= 16 && n % 4 == 0 && n >= 4 * (32 / rhs_bits)) {
        const int wide = 64 * (32 / rhs_bits);
        const int wide_tiles = (n + wide - 1) / wide;
        const long long waves = m_vec * 2 * ((wide_tiles + 1) / 2);
        if (waves >= 2048 && wide_tiles > 1 && wide_tiles != 3 &&
            (row_slots == 0 || row_slots >= wide_least_slots(rhs_bits, n, k, waves, wide_tiles, rows)))
            return 24;
    }
    // One dword of B per lane and one k-block of gathers in flight per wave:
    // latency is hidden by more resident waves rather than deeper per-wave
    // pipelines.  Up to four waves share a row (one per 16 * 32/bits
    // columns), and when the launch would hold fewer than 2048 waves (8 per
    // CU) the row's k-blocks are also split between two waves.  Measured on
    // MI355X over M = K = 4096, N in {128, 256, 512}, V in {2, 8}, sparsity
    // 0.7-0.98, every pair, and the reference's 2304-deep shapes: within 9 %
    // of the best tile everywhere (the autotuner covers the rest).
    // With eight or more column tiles and 4096 to 8191 waves, eight waves
    // share a row (one workgroup per row at n = 512 for 8-bit B).  Measured
    // on MI355X over M = K = 4096, N = 512, V in {2, 4, 8}, s in {0.7, 0.9,
    // 0.98} for L8-R8 and L16-R8: at V = 8 (4096 waves) within 1 % of the
    // best tile, 1-2 % better than four waves per row at s = 0.7 and 0.98;
    // at V = 2 and 4 (8192 waves and more) four waves per row are better
    // (3-6 % at s = 0.9), and two k-blocks in flight, best there at s <= 0.9,
    // lose 20-30 % at s = 0.98, where the rows are short.
    const int tile_cols = 16 * (32 / rhs_bits);
    const int tiles = (n + tile_cols - 1) / tile_cols;
    if (tiles >= 8) {
        const long long waves8 = m_vec * ((tiles + 7) / 8) * 8;
        if (waves8 >= 4096 && waves8 < 8192) return 13;
    }
    const int tpb = tiles >= 4 ? 4 : (tiles >= 2 ? 2 : 1);
    const long long waves = m_vec * ((tiles + tpb - 1) / tpb) * tpb;
    if (waves < 2048) return tpb == 4 ? 20 : 22;
    return tpb == 4 ? 17 : (tpb == 2 ? 16 : 15);
}

// Four dwords per lane are built for 8- and 16-bit B only (4-bit B would
// hold 32 accumulator tiles per wave); the B-stationary kernel is built for
// 8-bit B.
bool config_supported(int cfg, int rhs_bits) {
    if (kSpmmConfigs[cfg].kind == 1) return rhs_bits == 8;
    return rhs_bits != 4 || kSpmmConfigs[cfg].lane_dwords < 4;
}

// The reference's precision table (SpMM/SpMM/spmm_benchmark.cpp:805-831).
bool pair_supported(int lhs_bits, int rhs_bits) {
    switch (rhs_bits) {
    case 4: return lhs_bits == 4 || lhs_bits == 8 || lhs_bits == 12 || lhs_bits == 16;
    case 8: return lhs_bits == 8 || lhs_bits == 12 || lhs_bits == 16;
    case 16: return lhs_bits == 16;
    default: return false;
    }
}

mc_status spmm_entry(int lhs_bits, int rhs_bits, mc_signedness sign, int config, int m_vec, int vec_length, int n,
                     int k, const int *row_indices, const int *row_offsets, const int *column_indices,
                     const int *values, const int *rhs_matrix, int *output_matrix, hipStream_t stream,
                     int batch = 1, long long values_stride = 0, long long rhs_stride = 0,
                     long long out_stride = 0, __half *out16 = nullptr, float divisor = 1.f,
                     int row_slots = 0) {
    if (!pair_supported(lhs_bits, rhs_bits)) return MC_EUNSUPPORTED;
    if (batch < 1 || batch > 65535 || values_stride < 0 || rhs_stride < 0 || out_stride < 0) return MC_EINVAL_SHAPE;
    if ((values_stride | rhs_stride) & 3) return MC_EINVAL_SHAPE;   // every matrix starts dword aligned
    if (sign != MC_SIGNED && sign != MC_UNSIGNED) return MC_EINVAL_ARG;
    if (!valid_v(vec_length)) return MC_EINVAL_V;
    if (m_vec < 0 || n <= 0 || k <= 0) return MC_EINVAL_SHAPE;
    const int cpd = 32 / rhs_bits;
    if (n % cpd != 0) return MC_EINVAL_SHAPE;
    const long long rhs_bytes = (long long)k * n * rhs_bits / 8;
    if (rhs_bytes >= (1LL << 30)) return MC_EINVAL_SHAPE;   // gather offsets stay below 2^30
    if ((long long)m_vec * vec_length * (long long)n >= (1LL << 40)) return MC_EINVAL_SHAPE;
    if (m_vec == 0) return MC_OK;
    if (!row_offsets || !column_indices || !values || !rhs_matrix || !(output_matrix || out16)) return MC_EINVAL_ARG;
    if (config < -1 || config >= kNumSpmmConfigs) return MC_EINVAL_ARG;
    // a batched launch fills the GPU with (row, tile) x batch workgroups
    const int rows = out16 ? 32 : mfma_rows(lhs_bits, rhs_bits, sign == MC_SIGNED, vec_length);
    int cfg = config >= 0 ? config : default_config(rhs_bits, n, k, (long long)m_vec * batch, rows, row_slots);
    if (!config_supported(cfg, rhs_bits)) return MC_EUNSUPPORTED;
    if (batch > 1 && kSpmmConfigs[cfg].kind == 1) return MC_EUNSUPPORTED;   // B-stationary: one matrix
    if (kSpmmConfigs[cfg].kind == 1 && !stationary_fits(cfg, n, k)) {
        if (config >= 0) return MC_EINVAL_SHAPE;
        cfg = 7;   // the gather kernel takes any k
    }
    // an explicit tile's lanes divide a row; the default's last lane may
    // repeat columns of its neighbour
    if (config >= 0 && (n / cpd) % kSpmmConfigs[cfg].lane_dwords != 0) return MC_EINVAL_SHAPE;

    SpmmArgs a{};
    a.m_vec = m_vec;
    a.n = n;
    a.k = k;
    a.row_indices = row_indices;
    a.row_offsets = row_offsets;
    a.col_indices = column_indices;
    a.values = reinterpret_cast<const unsigned char *>(values);
    a.rhs = reinterpret_cast<const unsigned char *>(rhs_matrix);
    a.out = output_matrix;
    a.rhs_bytes = (unsigned)rhs_bytes;
    a.values_stride = values_stride;
    a.rhs_stride = rhs_stride;
    a.out_stride = out_stride;
    a.batch = batch;
    if (out16) {
        // 8-byte stores of four columns
        if ((reinterpret_cast<uintptr_t>(out16) & 7u) != 0 || (batch > 1 && out_stride % 4 != 0)) return MC_EINVAL_ARG;
        a.out16 = out16;
        a.div = make_divisor(divisor);
        return spmm_layer_launch_pair(lhs_bits, rhs_bits, vec_length, cfg, a, stream);
    }
    const bool sgn = sign == MC_SIGNED;
    if (lhs_bits == 8 && rhs_bits == 8) return spmm_launch_l8r8(sgn, vec_length, cfg, a, stream);
    if (lhs_bits == 16 && rhs_bits == 8) return spmm_launch_l16r8(sgn, vec_length, cfg, a, stream);
    if (lhs_bits == 12 && rhs_bits == 8) return spmm_launch_l12r8(sgn, vec_length, cfg, a, stream);
    if (lhs_bits == 16 && rhs_bits == 16) return spmm_launch_l16r16(sgn, vec_length, cfg, a, stream);
    if (lhs_bits == 8 && rhs_bits == 4) return spmm_launch_l8r4(sgn, vec_length, cfg, a, stream);
    if (lhs_bits == 12 && rhs_bits == 4) return spmm_launch_l12r4(sgn, vec_length, cfg, a, stream);
    if (lhs_bits == 16 && rhs_bits == 4) return spmm_launch_l16r4(sgn, vec_length, cfg, a, stream);
    return spmm_launch_l4r4(sgn, vec_length, cfg, a, stream);
}

}  // namespace
}  // namespace mc

extern "C" {

mc_status mc_spmm_l8r8(int m_vec, int vec_length, int n, int k, const int *row_indices, const int *row_offsets,
                       const int *column_indices, const int *values, const int *rhs_matrix, int *output_matrix,
                       mc_signedness sign, hipStream_t stream) {
    return mc::spmm_entry(8, 8, sign, -1, m_vec, vec_length, n, k, row_indices, row_offsets, column_indices, values,
                          rhs_matrix, output_matrix, stream);
}

mc_status mc_spmm_l16r8(int m_vec, int vec_length, int n, int k, const int *row_indices, const int *row_offsets,
                        const int *column_indices, const int *values, const int *rhs_matrix, int *output_matrix,
                        mc_signedness sign, hipStream_t stream) {
    return mc::spmm_entry(16, 8, sign, -1, m_vec, vec_length, n, k, row_indices, row_offsets, column_indices,
                          values, rhs_matrix, output_matrix, stream);
}

mc_status mc_spmm_l8r4(int m_vec, int vec_length, int n, int k, const int *row_indices, const int *row_offsets,
                       const int *column_indices, const int *values, const int *rhs_matrix, int *output_matrix,
                       mc_signedness sign, hipStream_t stream) {
    return mc::spmm_entry(8, 4, sign, -1, m_vec, vec_length, n, k, row_indices, row_offsets, column_indices, values,
                          rhs_matrix, output_matrix, stream);
}

mc_status mc_spmm_l4r4(int m_vec, int vec_length, int n, int k, const int *row_indices, const int *row_offsets,
                       const int *column_indices, const int *values, const int *rhs_matrix, int *output_matrix,
                       mc_signedness sign, hipStream_t stream) {
    return mc::spmm_entry(4, 4, sign, -1, m_vec, vec_length, n, k, row_indices, row_offsets, column_indices, values,
                          rhs_matrix, output_matrix, stream);
}

mc_status mc_spmm_l12r8(int m_vec, int vec_length, int n, int k, const int *row_indices, const int *row_offsets,
                       const int *column_indices, const int *values, const int *rhs_matrix, int *output_matrix,
                       mc_signedness sign, hipStream_t stream) {
    return mc::spmm_entry(12, 8, sign, -1, m_vec, vec_length, n, k, row_indices, row_offsets, column_indices, values,
                          rhs_matrix, output_matrix, stream);
}

mc_status mc_spmm_l16r16(int m_vec, int vec_length, int n, int k, const int *row_indices, const int *row_offsets,
                       const int *column_indices, const int *values, const int *rhs_matrix, int *output_matrix,
                       mc_signedness sign, hipStream_t stream) {
    return mc::spmm_entry(16, 16, sign, -1, m_vec, vec_length, n, k, row_indices, row_offsets, column_indices, values,
                          rhs_matrix, output_matrix, stream);
}

mc_status mc_spmm_l12r4(int m_vec, int vec_length, int n, int k, const int *row_indices, const int *row_offsets,
                       const int *column_indices, const int *values, const int *rhs_matrix, int *output_matrix,
                       mc_signedness sign, hipStream_t stream) {
    return mc::spmm_entry(12, 4, sign, -1, m_vec, vec_length, n, k, row_indices, row_offsets, column_indices, values,
                          rhs_matrix, output_matrix, stream);
}

mc_status mc_spmm_l16r4(int m_vec, int vec_length, int n, int k, const int *row_indices, const int *row_offsets,
                       const int *column_indices, const int *values, const int *rhs_matrix, int *output_matrix,
                       mc_signedness sign, hipStream_t stream) {
    return mc::spmm_entry(16, 4, sign, -1, m_vec, vec_length, n, k, row_indices, row_offsets, column_indices, values,
                          rhs_matrix, output_matrix, stream);
}

int mc_spmm_num_tile_configs(void) { return mc::kNumSpmmConfigs; }

mc_status mc_spmm_get_tile_config(int index, mc_tile_config *out) {
    if (index < 0 || index >= mc::kNumSpmmConfigs || !out) return MC_EINVAL_ARG;
    *out = mc::kSpmmConfigs[index];
    return MC_OK;
}

int mc_spmm_default_config(int lhs_bits, int rhs_bits, mc_signedness sign, int m_vec, int vec_length, int n, int k,
                           int row_slots) {
    if (!mc::pair_supported(lhs_bits, rhs_bits) || !mc::valid_v(vec_length) || m_vec < 0 || n <= 0 || k < 0 ||
        n % (32 / rhs_bits) != 0 || row_slots < 0)
        return -1;
    return mc::default_config(rhs_bits, n, k, m_vec, mc::mfma_rows(lhs_bits, rhs_bits, sign == MC_SIGNED, vec_length),
                              row_slots);
}

mc_status mc_spmm_run_rows(int lhs_bits, int rhs_bits, mc_signedness sign, int row_slots, int m_vec, int vec_length,
                           int n, int k, const int *row_indices, const int *row_offsets, const int *column_indices,
                           const int *values, const int *rhs_matrix, int *output_matrix, hipStream_t stream) {
    if (row_slots < 0) return MC_EINVAL_ARG;
    return mc::spmm_entry(lhs_bits, rhs_bits, sign, -1, m_vec, vec_length, n, k, row_indices, row_offsets,
                          column_indices, values, rhs_matrix, output_matrix, stream, 1, 0, 0, 0, nullptr, 1.f,
                          row_slots);
}

mc_status mc_spmm_run(int lhs_bits, int rhs_bits, mc_signedness sign, int config, int m_vec, int vec_length, int n,
                      int k, const int *row_indices, const int *row_offsets, const int *column_indices,
                      const int *values, const int *rhs_matrix, int *output_matrix, hipStream_t stream) {
    return mc::spmm_entry(lhs_bits, rhs_bits, sign, config, m_vec, vec_length, n, k, row_indices, row_offsets,
                          column_indices, values, rhs_matrix, output_matrix, stream);
}

mc_status mc_spmm_batched(int lhs_bits, int rhs_bits, mc_signedness sign, int config, int batch, int m_vec,
                          int vec_length, int n, int k, const int *row_indices, const int *row_offsets,
                          const int *column_indices, const int *values, long long values_stride_bytes,
                          const int *rhs_matrix, long long rhs_stride_bytes, int *output_matrix,
                          long long out_stride, hipStream_t stream) {
    return mc::spmm_entry(lhs_bits, rhs_bits, sign, config, m_vec, vec_length, n, k, row_indices, row_offsets,
                          column_indices, values, rhs_matrix, output_matrix, stream, batch, values_stride_bytes,
                          rhs_stride_bytes, out_stride);
}

mc_status mc_spmm_batched_f16(int lhs_bits, int rhs_bits, int batch, int m_vec, int vec_length, int n, int k,
                              const int *row_indices, const int *row_offsets, const int *column_indices,
                              const int *p, long long p_stride_bytes, const int *rhs_matrix,
                              long long rhs_stride_bytes, float divisor, void *out_f16, long long out_stride,
                              hipStream_t stream) {
    if (!((lhs_bits == 8 || lhs_bits == 16) && rhs_bits == 8) && !((lhs_bits == 8 || lhs_bits == 4) && rhs_bits == 4))
        return MC_EUNSUPPORTED;
    if (m_vec > 0 && !out_f16) return MC_EINVAL_ARG;
    return mc::spmm_entry(lhs_bits, rhs_bits, MC_SIGNED, -1, m_vec, vec_length, n, k, row_indices, row_offsets,
                          column_indices, p, rhs_matrix, nullptr, stream, batch, p_stride_bytes, rhs_stride_bytes,
                          out_stride, static_cast<__half *>(out_f16), divisor);
}

}  // extern "C"
