// plis_resident.h -- the host's view of the resident step kernel
// (plis_resident.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "plis_types.h"

namespace plis {

constexpr uint32_t kResidentQueue = 192;  // queued draws per wavefront
constexpr uint32_t kResidentMaxN = 16384; // subvolumes of a realization, whatever the network
constexpr uint32_t kResidentLdsMax = 160u * 1024u - 2048u;  // dynamic LDS, next to the kernel's own

struct ResidentArgs {
    KernelArgs k;
    uint32_t iters;         // iterations to make at most
    const int4* rx;         // reaction tables as ResTables describes them
    const int2 *sp, *spe, *jp, *jpe, *hm;
    uint32_t nspe;          // entries of spe and of jpe
    uint64_t diffusing;     // bit s: species s diffuses in some compartment
    const uint4* fwd;       // forward entries {upper end, weight, lower end, weight back}
    char* ws;               // global workspace, one slice per realization
    uint64_t ws_slice;      // bytes of a slice
};

// Bytes of dynamic LDS a block takes (the kernel lays it out in this order):
// queues, tile counters and tables; then the arrays; then the topology.
struct ResidentLds {
    uint64_t tables, arrays, topology;
};
inline ResidentLds resident_lds(uint64_t waves, uint64_t S, uint64_t R, uint64_t C, uint64_t nspe, uint64_t N,
                                uint64_t nf, uint64_t ne) {
    auto up = [](uint64_t b) { return (b + 15) & ~15ull; };
    ResidentLds l;
    l.tables = up(waves * kResidentQueue * 8) + up((N + 63) / 64 * 4) + up(C * R * 8) + up(C * S * 8) + up(R * 32) +
               2 * up(S * 8) + up(R * 8) + 2 * up(nspe * 8);
    l.arrays = up(N * (8 * R + 16 * S));
    l.topology = up(N * 8) + up(nf * 16) + up((N + 1) * 4) + up(ne * 8) + (C > 1 ? up(N * 4) : 0);
    return l;
}

// Lets the kernel take `lds` bytes of dynamic LDS.
hipError_t resident_reserve(uint32_t lds);

hipError_t launch_resident(hipStream_t stream, uint32_t nreal, uint32_t waves, uint32_t lds, int mode,
                           const ResidentArgs& a);

}  // namespace plis
