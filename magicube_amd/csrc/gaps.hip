// Zeroing of the slots between a vector-sparse mask's rows.
#include "mc_internal.hpp"

namespace mc {
namespace {

// Zeroes the slots that no row writes: row m's gap [start + roundup(nonzeros,
// group), start of row m + 1), the slots before row 0 and after the last row.
// slot_bits: bits a slot takes in the output.  Launched before the rows are
// written, so that any row order in memory is right (a gap that covers
// another row's slots is overwritten by that row; walking row by row from 0
// to the end crosses every slot in a row or in a gap).  A mask aligned to
// 16 or 32 slots leaves a few slots per row: 2 us, where filling the whole
// output takes 5.5 us for 27 MB of logits (8 heads, L = 4096, 90 % sparse).
__global__ __launch_bounds__(256) void zero_gaps_kernel(int m_vec, const int *row_offsets, int slots, int group,
                                                        int slot_bits, unsigned char *out, long long stride_bytes) {
    const int lane = threadIdx.x & 63, m = (int)(blockIdx.x * 4 + (threadIdx.x >> 6)) - 1;
    if (m >= m_vec) return;
    long long from = 0;
    if (m >= 0) {
        const int start = row_offsets[2 * m], end = row_offsets[2 * m + 1];
        from = (long long)start + (end - start + group - 1) / group * group;
    }
    const long long to = m + 1 < m_vec ? min(row_offsets[2 * (m + 1)], slots) : slots;
    unsigned char *o = out + blockIdx.y * stride_bytes;
    const long long b0 = from * slot_bits / 8, b1 = to * slot_bits / 8;
    if (((reinterpret_cast<uintptr_t>(o) | b0 | b1) & 3) == 0) {
        for (long long b = b0 + 4 * lane; b < b1; b += 256) *reinterpret_cast<int *>(o + b) = 0;
    } else {
        for (long long b = b0 + lane; b < b1; b += 64) o[b] = 0;
    }
}

}  // namespace

mc_status zero_gaps(int batch, int m_vec, const int *row_offsets, int slots, int group, int slot_bits, void *out,
                    long long stride_bytes, hipStream_t stream) {
    hipLaunchKernelGGL(zero_gaps_kernel, dim3((unsigned)(m_vec / 4 + 1), (unsigned)batch), dim3(256), 0, stream, m_vec,
                       row_offsets, slots, group, slot_bits, static_cast<unsigned char *>(out), stride_bytes);
    return check_launch();
}

}  // namespace mc
