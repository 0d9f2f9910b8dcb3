// plis_variant_learned.hip -- the learned-tau kernels of one (species,
// reactions) bound and their launches; compiled once per bound, like
// plis_variant.hip.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "plis_launch.h"
#include "plis_learned.hip"

namespace plis {

template <int MS, int MR>
void launch_learned(const LaunchEnv& c, int which, const KernelArgs& a) {
    const dim3 grid(c.blocks), block(64 * c.wpb);
    const bool mc = c.mc, gelu = c.gelu;
    // fewer, longer-lived blocks: each stages the network in LDS
    const dim3 fgrid(std::max<uint32_t>(8u, std::min<uint32_t>(c.blocks, (c.cus * c.finish_bpc + 7u) & ~7u)));
    const dim3 lgrid(std::max<uint32_t>(8u, std::min<uint32_t>(c.blocks, (c.cus * c.learned_bpc + 7u) & ~7u)));
    switch (which) {
        case kLearnedTau:
            // one pass covers fallbacks and refreshes; in steady state
            // it skips every tile, so it runs on a small grid
            if (mc && gelu) hipLaunchKernelGGL((learned_tau_kernel<MS, MR, true, 1>), lgrid, block, 0, c.stream, a);
            else if (mc) hipLaunchKernelGGL((learned_tau_kernel<MS, MR, true, 0>), lgrid, block, 0, c.stream, a);
            else if (gelu) hipLaunchKernelGGL((learned_tau_kernel<MS, MR, false, 1>), lgrid, block, 0, c.stream, a);
            else hipLaunchKernelGGL((learned_tau_kernel<MS, MR, false, 0>), lgrid, block, 0, c.stream, a);
            break;
        case kLearnedFinish:
            if (mc && gelu) hipLaunchKernelGGL((learned_finish_kernel<MS, MR, true, 1>), fgrid, block, 0, c.stream, a);
            else if (mc) hipLaunchKernelGGL((learned_finish_kernel<MS, MR, true, 0>), fgrid, block, 0, c.stream, a);
            else if (gelu) hipLaunchKernelGGL((learned_finish_kernel<MS, MR, false, 1>), fgrid, block, 0, c.stream, a);
            else hipLaunchKernelGGL((learned_finish_kernel<MS, MR, false, 0>), fgrid, block, 0, c.stream, a);
            break;
        case kLearnedRecords:
            hipLaunchKernelGGL((records_kernel<MS, MR>), grid, block, 0, c.stream, a);
            break;
        default:
            break;
    }
}

template void launch_learned<PLIS_MS, PLIS_MR>(const LaunchEnv&, int, const KernelArgs&);

}  // namespace plis
