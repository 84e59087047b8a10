// The selection kernels of forests whose nodes have at most 64 children.
#include "omk_select_kernels.h"

namespace omk {
template hipError_t launch_select_class<1, false>(const ForestDev &, const SelectArgs &, int, int, int, int,
                                                      const LoneOut &, hipStream_t);
template hipError_t launch_select_class<1, true>(const ForestDev &, const SelectArgs &, int, int, int, int,
                                                      const LoneOut &, hipStream_t);
}  // namespace omk
