// The wide GEMM tiles for int8 weights, bf16 activations (compiled in parallel with the other variants; see ql_gemm_wide.h).
#include "ql_gemm_wide.h"
namespace ql {
kern_t pick_wide_bf16_i8(int mt, int group, bool rope, bool alone) {
    return rope ? pick_wide_w16<false, true>(mt, group, alone) : pick_wide_w16<false, false>(mt, group, alone);
}
}  // namespace ql
