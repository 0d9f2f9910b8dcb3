// plis_variant.hip -- the step kernels of one (species, reactions) bound and
// their launches.  The build compiles this file once per bound (PLIS_MS and
// PLIS_MR given on the command line), in parallel.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "plis_launch.h"
#include "plis_learned.hip"

namespace plis {

// Kernel groups: 0 tau pass (learned and/or Cao), 1 decide, 2 leap pass,
// 3 commit; 4 tau pass on the counts the leap pass wrote and 6 commit +
// decide (the folded order of plain tau); 5 = training records of one
// realization.  In a learned
// context the end of the edge-parallel leap pass also proposes the next
// step's tau (learned_finish_kernel); learned_tau_kernel covers the steps
// whose proposals it could not make.
template <int MS, int MR>
void launch_variant(const LaunchEnv& c, int which, const KernelArgs& a) {
    const dim3 grid(c.blocks), block(64 * c.wpb), rgrid(c.nreal), rblock(1024), dblock(decide_threads<MS>());
    const dim3 dgrid(c.nreal * c.decide_chunks);
    const bool mc = c.mc;  // several compartments: per-subvolume rate tables
    const bool gelu = c.gelu;
    // learned kernels stage the network in LDS once per block: fewer, longer-lived blocks
    // the redo list is usually empty or short: two blocks per CU walk it
    const dim3 rgrid2(std::max<uint32_t>(8u, std::min<uint32_t>(c.blocks, (c.cus * 2u + 7u) & ~7u)));
    const dim3 fgrid(std::max<uint32_t>(8u, std::min<uint32_t>(c.blocks, (c.cus * c.finish_bpc + 7u) & ~7u)));
    const dim3 lgrid(std::max<uint32_t>(8u, std::min<uint32_t>(c.blocks, (c.cus * c.learned_bpc + 7u) & ~7u)));
    switch (which) {
        case 0:
            if constexpr (MS <= 8) {
                if (c.learned_on) {
                    // one pass covers fallbacks and refreshes; in steady state
                    // it skips every tile, so it runs on a small grid
                    if (mc && gelu) hipLaunchKernelGGL((learned_tau_kernel<MS, MR, true, 1>), lgrid, block, 0, c.stream, a);
                    else if (mc) hipLaunchKernelGGL((learned_tau_kernel<MS, MR, true, 0>), lgrid, block, 0, c.stream, a);
                    else if (gelu) hipLaunchKernelGGL((learned_tau_kernel<MS, MR, false, 1>), lgrid, block, 0, c.stream, a);
                    else hipLaunchKernelGGL((learned_tau_kernel<MS, MR, false, 0>), lgrid, block, 0, c.stream, a);
                    break;
                }
            }
            if (mc) hipLaunchKernelGGL((phase_a_kernel<MS, MR, true>), grid, block, 0, c.stream, a);
            else hipLaunchKernelGGL((phase_a_kernel<MS, MR, false>), grid, block, 0, c.stream, a);
            break;
        case 1:
            hipLaunchKernelGGL((decide_kernel<MS, MR>), dgrid, dblock, 0, c.stream, a);
            break;
        case 2:
            if constexpr (MS <= 8) {
                if (c.edge_parallel) {
                    if (mc) {
                        hipLaunchKernelGGL((phase_b_kernel<MS, MR, true, true>), grid, block, 0, c.stream, a);
                        if (c.split_ev) (void)hipEventRecord(c.split_ev[0], c.stream);
                        hipLaunchKernelGGL((phase_b_redo_kernel<MS, MR, true>), rgrid2, block, 0, c.stream, a);
                        if (c.split_ev) (void)hipEventRecord(c.split_ev[1], c.stream);
                        if (!c.learned_on)
                            hipLaunchKernelGGL((phase_b_finish_kernel<MS, MR, true>), grid, block, 0, c.stream, a);
                        else if (gelu)
                            hipLaunchKernelGGL((learned_finish_kernel<MS, MR, true, 1>), fgrid, block, 0, c.stream, a);
                        else
                            hipLaunchKernelGGL((learned_finish_kernel<MS, MR, true, 0>), fgrid, block, 0, c.stream, a);
                    } else {
                        hipLaunchKernelGGL((phase_b_kernel<MS, MR, true, false>), grid, block, 0, c.stream, a);
                        if (c.split_ev) (void)hipEventRecord(c.split_ev[0], c.stream);
                        hipLaunchKernelGGL((phase_b_redo_kernel<MS, MR, false>), rgrid2, block, 0, c.stream, a);
                        if (c.split_ev) (void)hipEventRecord(c.split_ev[1], c.stream);
                        if (!c.learned_on)
                            hipLaunchKernelGGL((phase_b_finish_kernel<MS, MR, false>), grid, block, 0, c.stream, a);
                        else if (gelu)
                            hipLaunchKernelGGL((learned_finish_kernel<MS, MR, false, 1>), fgrid, block, 0, c.stream, a);
                        else
                            hipLaunchKernelGGL((learned_finish_kernel<MS, MR, false, 0>), fgrid, block, 0, c.stream, a);
                    }
                    break;
                }
            }
            if (mc) hipLaunchKernelGGL((phase_b_kernel<MS, MR, false, true>), grid, block, 0, c.stream, a);
            else hipLaunchKernelGGL((phase_b_kernel<MS, MR, false, false>), grid, block, 0, c.stream, a);
            break;
        case 3:
            hipLaunchKernelGGL(commit_kernel, rgrid, rblock, 0, c.stream, a);
            break;
        case 4: {  // folded order: the tau pass on the counts the leap pass wrote
            KernelArgs as = a;
            as.tau_spec = 1u;
            if (mc) hipLaunchKernelGGL((phase_a_kernel<MS, MR, true>), grid, block, 0, c.stream, as);
            else hipLaunchKernelGGL((phase_a_kernel<MS, MR, false>), grid, block, 0, c.stream, as);
            break;
        }
        case 6:  // folded order: commit and decide
            hipLaunchKernelGGL((commit_decide_kernel<MS, MR>), dgrid, dblock, 0, c.stream, a);
            break;
        case 5:
            if constexpr (MS <= 8) hipLaunchKernelGGL((records_kernel<MS, MR>), grid, block, 0, c.stream, a);
            break;
        default:
            break;
    }
}

template void launch_variant<PLIS_MS, PLIS_MR>(const LaunchEnv&, int, const KernelArgs&);

}  // namespace plis
