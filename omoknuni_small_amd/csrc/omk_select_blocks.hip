// The selection kernels of batches with few visitors a root, by fan-out class.
#include "omk_select_blocks.h"

namespace omk {

template <int RMAX, bool RAVE>
static hipError_t launch_class(const ForestDev &f, const SelectArgs &a, int n_items, int n_singles, const LoneOut &out,
                               hipStream_t s) {
    const dim3 grid(n_items + (n_singles + kBlockWaves - 1) / kBlockWaves), block(kBlockWaves * kWave);
    if (out.sig.flag) hipLaunchKernelGGL((k_select_blocks<RMAX, RAVE, true>), grid, block, 0, s, f, a, n_items, n_singles, out);
    else hipLaunchKernelGGL((k_select_blocks<RMAX, RAVE, false>), grid, block, 0, s, f, a, n_items, n_singles, out);
    return hipGetLastError();
}

hipError_t launch_select_blocks(const ForestDev &f, const SelectArgs &a0, int n_items, int n_singles, int max_fanout, bool rave,
                                const LoneOut &out, hipStream_t s) {
    SelectArgs a = a0;
    if (!a.stats && !a.trace) a.times = nullptr;  // nobody has cleared them, nobody reads them
    if (max_fanout <= 64)
        return rave ? launch_class<1, true>(f, a, n_items, n_singles, out, s)
                    : launch_class<1, false>(f, a, n_items, n_singles, out, s);
    if (max_fanout <= 256)
        return rave ? launch_class<4, true>(f, a, n_items, n_singles, out, s)
                    : launch_class<4, false>(f, a, n_items, n_singles, out, s);
    return rave ? launch_class<6, true>(f, a, n_items, n_singles, out, s)
                : launch_class<6, false>(f, a, n_items, n_singles, out, s);
}

}  // namespace omk
