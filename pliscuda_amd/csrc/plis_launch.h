// plis_launch.h -- what the host side of the library and the translation
// units that hold its step kernels share.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "plis_types.h"

namespace plis {

// A context's launch shape and the switches that select kernels.
struct LaunchEnv {
    hipStream_t stream;
    hipEvent_t* split_ev;  // profiling: events between the leap pass's kernels, or nullptr
    uint32_t blocks, wpb, nreal, decide_chunks, cus, finish_bpc, learned_bpc;
    bool mc, asym, gelu, learned_on, edge_parallel;
    bool leap_split;  // a tile of the edge-parallel leap per block of 4 wavefronts
};

// decide_kernel and commit_decide_kernel: most blocks per realization
constexpr uint32_t kDecideChunks = 16;

// Launches one kernel group of the instantiation for at most MS species and
// MR reactions (plis_variant.hip).
template <int MS, int MR>
void launch_variant(const LaunchEnv& c, int which, const KernelArgs& a);

// The learned kernels of the instantiation (plis_variant_learned.hip; at most
// 8 species and 16 reactions).
enum LearnedKernel { kLearnedTau, kLearnedFinish, kLearnedRecords };
template <int MS, int MR>
void launch_learned(const LaunchEnv& c, int which, const KernelArgs& a);

}  // namespace plis
