// Gemm / MatMul on the f16 matrix cores (half_product.h holds the kernel and says what it computes).
#include "half_product.h"

namespace wdhc {
int launch_half_gemm(const HalfPlan &s, Params &p, const HalfOperand &w) {
  g_last_form = p.sB0 == 1 ? WDH_FORM_GEMM_KC : WDH_FORM_GEMM_MC;
  return launch_half<H_ROWS>(s, p, w);
}
}  // namespace wdhc
