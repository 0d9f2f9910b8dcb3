// plis_variant.hip -- the step kernels of one (species, reactions) bound and
// their launches.  The build compiles this file once per bound (PLIS_MS and
// PLIS_MR given on the command line), in parallel.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "plis_launch.h"
#include "plis_kernels.hip"

namespace plis {

// Kernel groups: 0 tau pass (learned and/or Cao), 1 decide, 2 leap pass,
// 3 commit; 4 tau pass on the counts the leap pass wrote and 6 commit +
// decide (the folded order of plain tau); 5 = training records of one
// realization; 7 = the target buffer before a call's first leap.  In a learned
// context the end of the edge-parallel leap pass also proposes the next
// step's tau (learned_finish_kernel); learned_tau_kernel covers the steps
// whose proposals it could not make.
template <int MS, int MR>
void launch_variant(const LaunchEnv& c, int which, const KernelArgs& a) {
    const dim3 grid(c.blocks), block(64 * c.wpb), rgrid(c.nreal), rblock(1024), dblock(decide_threads<MS>());
    const dim3 dgrid(c.nreal * c.decide_chunks);
    const bool mc = c.mc;  // several compartments: per-subvolume rate tables
    switch (which) {
        case 0:
            if constexpr (MS <= 8) {
                if (c.learned_on) {
                    launch_learned<MS, MR>(c, kLearnedTau, a);
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
                    const dim3 sgrid((a.ntiles + 7u) & ~7u), sblock(256);
                    const bool gen = mc || c.asym;
                    if (c.leap_split && gen) hipLaunchKernelGGL((phase_b_kernel<MS, MR, true, true, true>), sgrid, sblock, 0, c.stream, a);
                    else if (c.leap_split) hipLaunchKernelGGL((phase_b_kernel<MS, MR, true, false, true>), sgrid, sblock, 0, c.stream, a);
                    else if (gen) hipLaunchKernelGGL((phase_b_kernel<MS, MR, true, true, false>), grid, block, 0, c.stream, a);
                    else hipLaunchKernelGGL((phase_b_kernel<MS, MR, true, false, false>), grid, block, 0, c.stream, a);
                    if (c.split_ev) (void)hipEventRecord(*c.split_ev, c.stream);
                    if (c.learned_on) launch_learned<MS, MR>(c, kLearnedFinish, a);
                    else if (!a.judge_on) break;
                    else if (mc) hipLaunchKernelGGL((phase_b_finish_kernel<MS, MR, true>), grid, block, 0, c.stream, a);
                    else hipLaunchKernelGGL((phase_b_finish_kernel<MS, MR, false>), grid, block, 0, c.stream, a);
                    break;
                }
            }
            if (mc) hipLaunchKernelGGL((phase_b_kernel<MS, MR, false, true, false>), grid, block, 0, c.stream, a);
            else hipLaunchKernelGGL((phase_b_kernel<MS, MR, false, false, false>), grid, block, 0, c.stream, a);
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
        case 7:  // before a call's first step: the leap's target buffer
            hipLaunchKernelGGL(sync_target_kernel, grid, block, 0, c.stream, a);
            break;
        case 6:  // folded order: commit and decide
            hipLaunchKernelGGL((commit_decide_kernel<MS, MR>), dgrid, dblock, 0, c.stream, a);
            break;
        case 5:
            if constexpr (MS <= 8) launch_learned<MS, MR>(c, kLearnedRecords, a);
            break;
        default:
            break;
    }
}

template void launch_variant<PLIS_MS, PLIS_MR>(const LaunchEnv&, int, const KernelArgs&);

}  // namespace plis
