// Gemm / MatMul on the bf16 matrix cores (split_product.h holds the kernel and says what it computes).
#include "split_product.h"

namespace wdhc {
int launch_split_gemm(bool b_kc, const SplitPlan &s, Params &p, int nz) {
  return b_kc ? launch_split<B_KC>(s, p, nz) : launch_split<B_MC>(s, p, nz);
}
}  // namespace wdhc
