// The attention layer's P V products, fp16 out: signed, one tile per default
// of the SpMM family (see spmm_dispatch.hpp).
#include "spmm_dispatch.hpp"

namespace mc {
mc_status spmm_layer_launch_pair(int lhs_bits, int rhs_bits, int V, int cfg, const SpmmArgs &a, hipStream_t s) {
    if (lhs_bits == 8 && rhs_bits == 8) return spmm_layer_launch<8, 8>(V, cfg, a, s);
    if (lhs_bits == 16 && rhs_bits == 8) return spmm_layer_launch<16, 8>(V, cfg, a, s);
    if (lhs_bits == 8 && rhs_bits == 4) return spmm_layer_launch<8, 4>(V, cfg, a, s);
    if (lhs_bits == 4 && rhs_bits == 4) return spmm_layer_launch<4, 4>(V, cfg, a, s);
    return MC_EUNSUPPORTED;
}
}  // namespace mc
