// plis_dispatch.h -- the rules by which a context chooses its way of stepping.
// Plain host code: no HIP, so that a program without a GPU can evaluate them.
#pragma once
#include <stdint.h>

#include <algorithm>
#include <functional>
#include <queue>
#include <vector>

namespace plis {

// What a rule needs to know of a realization.
struct StepSize {
    uint64_t N, n_in, ntiles;  // subvolumes, in-edges, tiles of 64 subvolumes
};

// us that one CU's phases of a step take beyond their fixed latency.
inline double resident_phases_us(int S, int R, const StepSize& r) {
    return 1e-3 * ((double)r.N * (2.0 + 2.8 * R) + 0.84 * S * (double)r.n_in);
}

// Blocks of resident_kernel that a CU holds: its 128 registers a lane leave 16
// wavefronts, and 160 KB of LDS are shared (2 KB: the kernel's static part).
inline uint64_t resident_blocks_per_cu(uint32_t waves, uint32_t lds) {
    return std::max<uint64_t>(1, std::min<uint64_t>(16u / std::max(1u, waves), 160u * 1024u / (lds + 2048u)));
}

// us of an iteration of a context whose realizations step in one block each,
// `slots` of them at a time: every realization goes to the slot that is free
// first.  8 us + 0.6 of the phases with the chip full (6.5 us with one
// reaction; 257 against 256 realizations, measured: A-B-C 8^3 29.0 / 16.2 us,
// bistable 9^3 36.3 / 20.0, Brusselator mesh of 216 25.4 / 14.0).
inline double resident_step_us(int S, int R, const std::vector<StepSize>& rs, uint64_t slots) {
    const double base = std::min(8.0, 6.0 + 0.5 * R);
    std::priority_queue<double, std::vector<double>, std::greater<double>> busy;  // when a slot is free again
    double end = 0.0;
    for (const StepSize& r : rs) {
        double t = base + 0.6 * resident_phases_us(S, R, r);
        if (busy.size() >= slots) {
            t += busy.top();
            busy.pop();
        }
        busy.push(t);
        end = std::max(end, t);
    }
    return end;
}

// Whether realizations of these sizes step faster in one block each than with a
// launch per pass.  general: the step kernels are the general instantiation (more
// than 8 species or 16 reactions).
//
// One CU makes a step of N subvolumes in about 5 us + N (2 + 0.84 S deg +
// 2.8 R) ns (measured: A-B-C 7.6 us at 64, 15 at 512, 26 at 1,000, 41 at
// 1,728; diffusion of one species 21 at 1,728; Brusselator mesh 25 at 512,
// 50 at 1,000).  The launch-per-pass step takes 18 us with one species, 22
// with the three of A-B-C and 30 with the Brusselator's five at these sizes
// (both sides measured: bistable 18.7 / 19.1 us at 729; A-B-C 19.3 / 21.9
// at 729, 25.4 / 21.9 at 1,000; diffusion 14.1 / 18.0 at 1,000, 20.1 / 18.9
// at 1,728; Brusselator 23.5 / 29.8 at 512), and 680 us or more in its
// general instantiation (cascade of 32 species, 62 reactions: 17 us here at
// 60 subvolumes, 165 at 1,000).  The line lies where the two meet.
//
// More realizations than the chip holds blocks step in rounds, while the
// launches fill up with tiles: 14 + 3 S + tiles (2.3 + (S + R) / 2) / 1,000 us
// (measured, one block each / launch per pass: bistable 6^3, 512 realizations
// 24.4 / 27.1, 1,024 47.3 / 33.2, 3,000 143 / 86; A-B-C 6^3, 1,024 37.2 / 39.4,
// 3,000 109 / 90; diffusion 5^3, 1,024 15.4 / 22.8, 4,096 71.2 / 62.7; 8 species
// and 12 reactions on 64 subvolumes, 1,024 43 / 50, 2,048 85 / 61).  The general
// instantiation stays slower however many there are (the cascade on 60, 4,096
// realizations: 400 / 3,575).
inline bool resident_pays(int S, int R, bool general, const std::vector<StepSize>& rs, uint64_t slots) {
    double longest = 0.0;
    uint64_t tiles = 0;
    for (const StepSize& r : rs) {
        longest = std::max(longest, resident_phases_us(S, R, r));
        tiles += r.ntiles;
    }
    if (longest > (general ? 600.0 : 10.5 + 4.0 * S)) return false;
    if (general || rs.size() <= slots) return true;
    return resident_step_us(S, R, rs, slots) <= 14.0 + 3.0 * S + 1e-3 * (double)tiles * (2.3 + 0.5 * (S + R));
}

// Iterations of one launch that make `us` an iteration: some 50 ms, so that the
// host sees the realizations' progress and a wait for the stream stays short
// (4,096 at the general line of 600 us would take 2.5 s).  At most 1,024, which
// the smallest boxes make in 8 ms.
inline uint32_t resident_launch_iters(double us) {
    return (uint32_t)std::min(1024.0, std::max(1.0, 50e3 / us));
}

}  // namespace plis
