// The wide GEMM tiles for fp8 weights, bf16 activations (compiled in parallel with the other variants; see ql_gemm_wide.h).
#include "ql_gemm_wide.h"
namespace ql {
kern_t pick_wide_bf16_fp8(int mt, int group, bool rope, bool alone) {
    return rope ? pick_wide_w16<true, true>(mt, group, alone) : pick_wide_w16<true, false>(mt, group, alone);
}
}  // namespace ql
