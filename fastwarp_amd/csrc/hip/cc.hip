// The CC kernels of one window radius (FW_CC_RADIUS, 1 to 8), compiled once for each.
#include "cc_kernels.hpp"

#ifndef FW_CC_RADIUS
#error "FW_CC_RADIUS is the radius this object holds"
#endif

namespace fw::hip {

template void launch_cc_radius<FW_CC_RADIUS>(const CcArgs& a, hipStream_t s);
template void launch_cc_items_radius<FW_CC_RADIUS>(const CcItems& c, hipStream_t s);

}  // namespace fw::hip
