// Instantiates the fused dequant GEMM kernels for one arithmetic variant (compiled in parallel with
// the other variants; see ql_gemm_kernel.h).
#include "ql_gemm_kernel.h"
namespace ql {
kern_t pick_bf16_i8_row(int mt, int wn, int wk, int cp, bool rope) { return pick_kernel_impl<ACT_BF16, false, false>(mt, wn, wk, cp, rope); }
kern_t pick_bf16_i8_row_stop(int wn) {
    return wn == 1 ? (kern_t)qgemm_kernel<ACT_BF16, false, 1, 1, 8, 4, false, false, false, false, false, false, false, true>
                   : (kern_t)qgemm_kernel<ACT_BF16, false, 1, 2, 4, 8, false, false, false, false, false, false, false, true>;
}
}  // namespace ql
