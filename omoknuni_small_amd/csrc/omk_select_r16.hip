// The selection kernels of forests whose nodes have up to OMK_MAX_FANOUT children.
#include "omk_select_kernels.h"

namespace omk {
template hipError_t launch_select_class<16, false>(const ForestDev &, const SelectArgs &, int, int, int, int,
                                                      const LoneOut &, hipStream_t);
template hipError_t launch_select_class<16, true>(const ForestDev &, const SelectArgs &, int, int, int, int,
                                                      const LoneOut &, hipStream_t);
}  // namespace omk
