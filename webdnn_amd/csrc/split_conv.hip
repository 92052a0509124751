// Conv on the bf16 matrix cores (split_product.h holds the kernel and says what it computes).
#include "split_product.h"

namespace wdhc {
int launch_split_conv(int mode, const SplitPlan &s, Params &p, int nz) {
  switch (mode) {
    case B_PIXELS: return launch_split<B_PIXELS>(s, p, nz);
    case B_PIXELS_ANY: return launch_split<B_PIXELS_ANY>(s, p, nz);
    case B_IM2COL64: return launch_split<B_IM2COL64>(s, p, nz);
    default: return launch_split<B_IM2COL32>(s, p, nz);
  }
}
}  // namespace wdhc
