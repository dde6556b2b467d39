// The wide GEMM tiles for 8-bit weights and activations (compiled in parallel with the other variants; see ql_gemm_wide.h).
#include "ql_gemm_wide.h"
namespace ql {
kern_t pick_wide_i8_i8(int mt, bool rope) { return rope ? pick_wide_impl<ACT_I8, false, 0, true>(mt) : pick_wide_impl<ACT_I8, false, 0, false>(mt); }
kern_t pick_wide_fp8_fp8(int mt, bool rope) { return rope ? pick_wide_impl<ACT_FP8, true, 0, true>(mt) : pick_wide_impl<ACT_FP8, true, 0, false>(mt); }
}  // namespace ql
