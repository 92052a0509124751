// 1x1 Conv on the f16 matrix cores (half_product.h holds the kernel and says what it computes).
#include "half_product.h"

namespace wdhc {
int launch_half_conv(const HalfPlan &s, Params &p, const HalfOperand &w) { return launch_half<H_PIXELS>(s, p, w); }
}  // namespace wdhc
