// The CC kernels of one window radius (FW_CC_RADIUS, 1 to 8) and one launch (FW_CC_PART: 0 a pair, 1 a pair with
// a mask, 2 the pairs of a batch), compiled once for each.
#include "cc_kernels.hpp"

#if !defined(FW_CC_RADIUS) || !defined(FW_CC_PART)
#error "FW_CC_RADIUS and FW_CC_PART say what this object holds"
#endif

namespace fw::hip {

#if FW_CC_PART == 2
template void launch_cc_items_radius<FW_CC_RADIUS>(const CcItems& c, hipStream_t s);
#else
template void launch_cc_radius<FW_CC_RADIUS, FW_CC_PART == 1>(const CcArgs& a, hipStream_t s);
#endif

}  // namespace fw::hip
