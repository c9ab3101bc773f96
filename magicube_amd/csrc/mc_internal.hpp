// Host-side helpers shared by the library's translation units.
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/magicube_hip.h"

namespace mc {

// Records a HIP failure for mc_last_hip_error() and maps it to MC_EHIP.
mc_status hip_fail(hipError_t e);

inline mc_status check_launch() {
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? MC_OK : hip_fail(e);
}

// Zeroes the output slots outside every row's [start, start + roundup(nonzeros,
// group)), up to `slots`, of each of `batch` matrices (gaps.hip); launched
// before the rows are written.
mc_status zero_gaps(int batch, int m_vec, const int *row_offsets, int slots, int group, int slot_bits, void *out,
                    long long stride_bytes, hipStream_t stream);

inline bool valid_v(int v) { return v == 2 || v == 4 || v == 8; }

}  // namespace mc
