// mixed_resident_fp16.hip -- the resident inner iterations with FP16 weights.
#include "mixed_resident.hpp"

namespace eafp {
int rmx_launch_fp16(bool line, int cq, int slots, const RMxArgs& g, int blocks, size_t lds, hipStream_t st) {
    return rmx_launch<EAFP_COEF_FP16>(line, cq, slots, g, blocks, lds, st);
}
int rmx_prepare_fp16(bool line, int cq, int slots) { return rmx_prepare<EAFP_COEF_FP16>(line, cq, slots); }
}  // namespace eafp
