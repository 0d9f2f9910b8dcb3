// plis_kernels.hip -- gfx950 kernels for the RDME tau-leap + SSA step.
//
// One global step of one realization is three kernels:
//   the leap (phase_b_kernel): Poisson firings of non-critical reactions and
//     hops, every linked pair drawn once by the tile of its lower end from a
//     counter-based Philox draw, integer balances added to a copy of the
//     counts, and the critical event.  Replaces leap_step (leap.cu:3-201) and
//     ssa_step (ssa.cu:56-110).
//   the tau pass on the counts the leap wrote (phase_a_kernel): per subvolume
//     FP64 mass-action propensities, Cao tau' with hops treated as first-order
//     channels, the critical set and an exponential tau'' clock, min / argmin
//     per 64-subvolume tile as a tile partial; and the range check of the new
//     counts (check_state + none_of, leap.cu:203-212, driver.cu:292-323).
//     Replaces compute_rates (PLISCuda/src/rates.cu:82-96) and compute_taus
//     (tau.cu:197-251).
//   commit_decide_kernel: reduces the partials, commits the step or leaps back
//     (tau' halved, new attempt index) and decides the next one.  Replaces the
//     host's thrust::min_element + tau[i] round trips and the revert
//     (driver.cu:267-277, 292-323).
//
// Wavefront-per-tile: lane i of a wave owns subvolume v0+i of its tile;
// species-major counts make every per-species load and store one coalesced
// 256-byte access.  Blocks are dispatched round-robin over the 8 XCDs, so
// each XCD walks a contiguous eighth of the tile list (its L2 holds the
// neighbouring tiles it gathers from).
#pragma once
#include <type_traits>

#include "plis_launch.h"
#include "plis_numerics.h"
#include "plis_types.h"

namespace plis {

constexpr double kInf = __builtin_huge_val();

// The network tables are read-only for every kernel: reading them through
// the constant address space lets the compiler use scalar loads (scalar
// cache, no vector-memory round trip) wherever the index is wave-uniform.
template <class T>
using cptr = const T __attribute__((address_space(4)))*;

// Per-kernel read-only data (tile table, realization info and control)
// through the same address space.
template <class T>
__device__ __forceinline__ cptr<T> ro(const T* p) {
    return (cptr<T>)p;
}

// A whole read-only struct, word by word (merged into wide scalar loads).
template <class T>
__device__ __forceinline__ T ld_ro(const T* p) {
    static_assert(sizeof(T) % 4 == 0, "struct of 32-bit words");
    T v;
    uint32_t* d = reinterpret_cast<uint32_t*>(&v);
    const cptr<uint32_t> w = (cptr<uint32_t>)p;
#pragma unroll
    for (int i = 0; i < (int)(sizeof(T) / 4); ++i) d[i] = w[i];
    return v;
}

struct NetView {
    cptr<int32_t> nu, rs, rr, nrs, order, hor, mult;
    cptr<double> k, d;
    int S, R, C;
};

// MC = false: the network has one compartment, known at compile time, so
// every compartment lookup folds to 0 and the rate constants and diffusion
// constants become wave-uniform (scalar) loads.
template <bool MC = true>
__device__ __forceinline__ NetView net_view(const KernelArgs& a) {
    NetView n;
    n.nu = (cptr<int32_t>)(a.net_i + a.nh.off_nu);
    n.rs = (cptr<int32_t>)(a.net_i + a.nh.off_rs);
    n.rr = (cptr<int32_t>)(a.net_i + a.nh.off_rr);
    n.nrs = (cptr<int32_t>)(a.net_i + a.nh.off_nrs);
    n.order = (cptr<int32_t>)(a.net_i + a.nh.off_order);
    n.hor = (cptr<int32_t>)(a.net_i + a.nh.off_hor);
    n.mult = (cptr<int32_t>)(a.net_i + a.nh.off_mult);
    n.k = (cptr<double>)(a.net_d + a.nh.off_k);
    n.d = (cptr<double>)(a.net_d + a.nh.off_d);
    n.S = a.nh.S;
    n.R = a.nh.R;
    n.C = MC ? a.nh.C : 1;
    return n;
}

__device__ __forceinline__ uint32_t wave_uniform(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}

// The kernel's arguments (its only parameter) through a pointer made opaque
// per tile: they and the network tables are loaded where a tile's work uses
// them instead of being hoisted out of the tile loop into (spilled) scalar
// registers.
__device__ __forceinline__ const KernelArgs& tile_args() {
    cptr<KernelArgs> p = (cptr<KernelArgs>)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const KernelArgs*)p;
}

// Orders one wavefront's LDS writes before its later LDS reads.
__device__ __forceinline__ void lds_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}


// XCD-aware persistent tile walk (grid is a multiple of 8 blocks).
__device__ __forceinline__ uint32_t tile_at(uint32_t it, uint32_t ntiles, uint32_t wpb, uint32_t wv) {
    const uint32_t G = gridDim.x;
    const uint32_t b = blockIdx.x;
    const uint32_t xcd = b & 7u;
    const uint32_t nbx = (G - xcd + 7u) >> 3;
    const uint32_t lb = b >> 3;
    const uint32_t cb = (uint32_t)(((uint64_t)ntiles * xcd) >> 3);
    const uint32_t ce = (uint32_t)(((uint64_t)ntiles * (xcd + 1u)) >> 3);
    const uint32_t t = cb + lb * wpb + wv + it * nbx * wpb;
    return t < ce ? t : 0xFFFFFFFFu;
}
__device__ __forceinline__ uint32_t tile_at(uint32_t it, uint32_t ntiles, uint32_t wpb) {
    return tile_at(it, ntiles, wpb, wave_uniform(threadIdx.x >> 6));
}

__device__ __forceinline__ uint32_t* count_buf(const KernelArgs& a, uint32_t i) {
    return a.x + (uint64_t)i * a.x_stride;
}

// The two count buffers that are neither the current nor the target one, in
// ascending order: the pass after an edge-parallel leap copies the new counts
// to the first and the old ones to the second.
__device__ __forceinline__ void spare_bufs(uint32_t cur, uint32_t tgt, uint32_t& z, uint32_t& w) {
    const uint32_t rest = 0xFu & ~(1u << cur) & ~(1u << tgt);
    z = (uint32_t)__builtin_ctz(rest);
    w = 31u - (uint32_t)__builtin_clz(rest);
}

// an interleaved edge entry's high word for weight 1.0 (a padding entry)
constexpr uint64_t kOneW = (uint64_t)0x3F800000u << 32;

__device__ __forceinline__ double binom_d(uint32_t x, int r) {
    if (x < (uint32_t)r) return 0.0;  // r >= 1
    const double xd = (double)x;
    if (r == 1) return xd;
    if (r == 2) return (xd * (xd - 1.0)) * 0.5;
    return ((xd * (xd - 1.0)) * (xd - 2.0)) / 6.0;
}

// Cao's critical test of one reactant, floor(x / r) < n_c, as the
// equivalent x < n_c r (integers, r >= 1, n_c >= 0): no division; n_c r is
// formed in 64 bits from scalars, one 64-bit compare per lane.
__device__ __forceinline__ bool below_nc(uint32_t x, int r, int nc) {
    return (uint64_t)x < (uint64_t)(uint32_t)nc * (uint64_t)(uint32_t)r;
}

// A hop is active (non-critical) when d > 0 and x >= max(n_c, 1).
__device__ __forceinline__ bool hop_active(double d, uint32_t x, int nc) {
    return d > 0.0 && x >= (uint32_t)(nc > 1 ? nc : 1);
}

__device__ __forceinline__ double g_cao(int hor, int mult, uint32_t xs) {
    const double xd = (double)xs;
    if (hor == 1) return 1.0;
    if (hor == 2) return mult == 2 ? 2.0 + 1.0 / (xd - 1.0) : 2.0;
    if (mult == 3) return (3.0 + 1.0 / (xd - 1.0)) + 2.0 / (xd - 2.0);
    if (mult == 2) return 1.5 * (2.0 + 1.0 / (xd - 1.0));
    return 3.0;
}

// eps x / g(x): for g = 1 and g = 2 (first order; second order with one
// molecule of the species) the quotient is formed without a divide -- x / 1
// and x / 2 are exact, so the result is the same IEEE value.
__device__ __forceinline__ double eps_x_over_g(double eps, int hor, int mult, uint32_t xs) {
    const double ex = eps * (double)xs;
    if (hor == 1) return ex;
    if (hor == 2 && mult != 2) return ex * 0.5;
    return ex / g_cao(hor, mult, xs);
}

// Reaction propensities a_j = k_j prod_s C(x_s, r_sj) and the critical flags
// (Cao: L_j = min_s floor(x_s / r_sj) < n_c, i.e. some reactant has
// floor(x_s / r_sj) < n_c) at one subvolume.
template <int MR, int MS>
__device__ __forceinline__ void react_props(const NetView& n, const uint32_t (&x)[MS], int c, int nc,
                                            double (&av)[MR], uint32_t (&crit)[(MR + 31) / 32]) {
#pragma unroll
    for (int i = 0; i < (MR + 31) / 32; ++i) crit[i] = 0u;
#pragma unroll
    for (int j = 0; j < MR; ++j) {
        if (j >= n.R) break;
        double aj = n.k[c * n.R + j];
        bool low = false;
        const int nr = n.nrs[j];
        for (int i = 0; i < nr; ++i) {
            const int s = n.rs[j * 3 + i], r = n.rr[j * 3 + i];
            uint32_t xs = 0;
#pragma unroll
            for (int q = 0; q < MS; ++q)
                if (q == s) xs = x[q];
            aj = aj * binom_d(xs, r);
            low = low || below_nc(xs, r, nc);
        }
        av[j] = aj;
        if (n.order[j] > 0 && low) crit[j >> 5] |= 1u << (j & 31);
    }
}

template <int MR>
__device__ __forceinline__ bool is_crit(const uint32_t (&crit)[(MR + 31) / 32], int j) {
    return (crit[j >> 5] >> (j & 31)) & 1u;
}

// Post-leap leap condition in propensity form (Cao, Gillespie & Petzold
// 2006, eq. 5, with their one-molecule floor; checked after the leap as in
// Anderson 2008).  A non-critical channel j with a_j(x) > 0 breaks it when
//     |a_j(x') - a_j(x)| > theta max(eps, phi_j) a_j(x),
// phi_j = max over reactants i of r_ij / x_i (one molecule's relative
// effect); evaluated without divides as D > (theta a_j) eps and
// D x_i > (theta a_j) r_ij for every reactant i.  An active hop channel of
// species s breaks it when |x'_s - x_s| > theta max(eps x_s, 1).  Bounds
// carry a relative slack of 2^-30 so that a change meeting one exactly (a
// one-molecule change at the floor) holds whatever the rounding of the
// products.  A negative or overflowing count breaks it too.  av / crit:
// propensities and critical flags of x.
constexpr double kLcSlack = 1.0 + 0x1p-30;
// av_new: a_j(x') when the caller has it (same operations, same values),
// else nullptr and the products are formed here.
template <int MS, int MR>
__device__ __forceinline__ uint32_t leap_condition_broken(const NetView& n, int c, int nc, double eps, double theta,
                                                          const uint32_t (&x)[MS], const long long (&nx)[MS],
                                                          const double (&av)[MR],
                                                          const uint32_t (&crit)[(MR + 31) / 32],
                                                          const double* av_new = nullptr) {
    uint32_t xn[MS];
    bool neg = false;
#pragma unroll
    for (int s = 0; s < MS; ++s) {
        neg = neg || (s < n.S && (nx[s] < 0 || nx[s] > 0xFFFFFFFFll));
        xn[s] = (uint32_t)nx[s];
    }
    if (neg) return 1u;
    uint32_t broken = 0u;
#pragma unroll
    for (int j = 0; j < MR; ++j) {
        if (j >= n.R) break;
        const int nr = n.nrs[j];
        if (is_crit<MR>(crit, j) || !(av[j] > 0.0) || nr == 0) continue;
        double aj;
        if (av_new) {
            aj = av_new[j];
        } else {
            aj = n.k[c * n.R + j];
            for (int i = 0; i < nr; ++i) {
                const int sp = n.rs[j * 3 + i], r = n.rr[j * 3 + i];
                uint32_t xs = 0;
#pragma unroll
                for (int q = 0; q < MS; ++q)
                    if (q == sp) xs = xn[q];
                aj = aj * binom_d(xs, r);
            }
        }
        const double D = __builtin_fabs(aj - av[j]);
        const double t = (theta * av[j]) * kLcSlack;
        bool over = D > t * eps;
        for (int i = 0; i < nr; ++i) {
            const int sp = n.rs[j * 3 + i], r = n.rr[j * 3 + i];
            uint32_t xs = 0;
#pragma unroll
            for (int q = 0; q < MS; ++q)
                if (q == sp) xs = x[q];
            over = over && D * (double)xs > t * (double)r;
        }
        if (over) broken = 1u;
    }
#pragma unroll
    for (int s = 0; s < MS; ++s) {
        if (s >= n.S) break;
        if (!hop_active(n.d[c * n.S + s], x[s], nc)) continue;
        if (__builtin_fabs((double)xn[s] - (double)x[s]) > (theta * fmax(eps * (double)x[s], 1.0)) * kLcSlack)
            broken = 1u;
    }
    return broken;
}

// ---------------------------------------------------------------------------
// per-realization step decision (tau = min(tau', tau''), clamp to t_end)
// ---------------------------------------------------------------------------
__device__ __forceinline__ void decide(RealCtl& c) {
    double tau = fmin(c.tau_p, c.tau2);
    c.crit = (c.tau2 <= c.tau_p) ? 1 : 0;
    c.last = 0;
    if (c.t + tau >= c.t_end) {
        tau = c.t_end - c.t;
        c.crit = 0;
        c.last = 1;
    }
    c.tau = tau;
}

// Destination of a critical hop from v: the edge of v's row at which the
// weights, summed one edge at a time in CSR order, pass tw.  Run by a whole
// wavefront, which loads up to 64 edges at once; cw: the first ones of the row
// [rb, re), from hop_row.
__device__ __forceinline__ uint32_t choose_hop_edge(const KernelArgs& a, const RealInfo& ri, uint32_t v, uint32_t rb,
                                                    uint32_t re, uint64_t cw, double tw) {
    const uint32_t lane = threadIdx.x & 63u;
    double accw = 0.0;
    uint32_t dst = v;
    bool found = false;
    for (uint32_t q0 = rb; q0 < re && !found; q0 += 64u) {
        if (q0 != rb) cw = a.cw[ri.e_off + min(q0 + lane, re - 1u)];
        const uint32_t cnt = min(64u, re - q0);
        for (uint32_t i = 0; i < cnt; ++i) {
            accw += (double)__int_as_float(__builtin_amdgcn_readlane((int)(cw >> 32), (int)i));
            dst = (uint32_t)__builtin_amdgcn_readlane((int)cw, (int)i);
            if (tw < accw) {
                found = true;
                break;
            }
        }
    }
    return dst;
}

// v's out-edges: the row's bounds and the lane's edge {id, weight} among the
// first 64.
struct HopRow {
    uint32_t rb, re;
    uint64_t cw;
};
__device__ __forceinline__ HopRow hop_row(const KernelArgs& a, const RealInfo& ri, uint32_t v) {
    HopRow h;
    h.rb = a.rp[ri.rp_off + v];
    h.re = a.rp[ri.rp_off + v + 1];
    h.cw = h.rb < h.re ? a.cw[ri.e_off + min(h.rb + (threadIdx.x & 63u), h.re - 1u)] : (uint64_t)v;
    return h;
}

__device__ __forceinline__ double lane_f64(double x, uint32_t l) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, (int)l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), (int)l);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Critical event at v*: a critical reaction or a critical hop, chosen with
// probability proportional to its propensity; a hop's edge is chosen in
// proportion to its weight.  (The reference picks a uniform slot among 6
// including self-padding, PLISCuda/src/leap.cu:180-194, ssa.cu:88-106.)
//
// Run by a whole wavefront: lane s takes species s, lane j reactions j and
// j + 64, so that every table entry is requested at once, and the sums then go
// over the lanes in the network's order, as one lane would form them.  (One
// reaction after the other, each waiting for its own table entries,
// commit_decide_kernel took 10.7 us on the 1M-subvolume Brusselator mesh, 8.9
// now, and 8.5 on 32 meshes in one context, 6.9 now.)
static __device__ void choose_event(const KernelArgs& a, const RealInfo& ri, RealCtl& c, const uint32_t* X) {
    const uint32_t v = c.vstar, lane = threadIdx.x & 63u;
    const int S = a.nh.S, R = a.nh.R, nc = a.n_critical;
    const int cc = a.nh.C > 1 ? a.comp[ri.comp_off + v] : 0;
    const double W = a.wsum[ri.rp_off + v];
    HopRow row = hop_row(a, ri, v);
    const int s = min((int)lane, S - 1);  // (kMaxS = 64 species, one a lane)
    const uint32_t xs = X[ri.x_off + (uint64_t)s * ri.N + v];
    const double d = a.net_d[a.nh.off_d + cc * S + s];
    const uint64_t hops = __ballot((int)lane < S && d > 0.0 && !hop_active(d, xs, nc));
    const double ao = (d * (double)xs) * W;
    double aj[2];
    uint64_t crit[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {  // (kMaxR = 128 reactions)
        const int j = min((int)lane + 64 * h, R > 0 ? R - 1 : 0);
        const bool on = (int)lane + 64 * h < R;
        const int nr = on ? a.net_i[a.nh.off_nrs + j] : 0, order = on ? a.net_i[a.nh.off_order + j] : 0;
        int sp[3], mu[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            sp[i] = on ? a.net_i[a.nh.off_rs + 3 * j + i] : 0;
            mu[i] = on ? a.net_i[a.nh.off_rr + 3 * j + i] : 1;
        }
        aj[h] = on ? a.net_d[a.nh.off_k + cc * R + j] : 0.0;
        bool low = false;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const uint32_t x = (uint32_t)__shfl((int)xs, i < nr ? sp[i] : 0);
            if (i >= nr) continue;
            aj[h] = aj[h] * binom_d(x, mu[i]);
            low = low || below_nc(x, mu[i], nc);
        }
        crit[h] = __ballot(on && order > 0 && low);
    }
    asm volatile("" : "+v"(row.cw));  // (loaded by now, not after the choice)
    double a0c = 0.0;
#pragma unroll
    for (int h = 0; h < 2; ++h)
        for (uint64_t m = crit[h]; m != 0ull; m &= m - 1ull) a0c += lane_f64(aj[h], (uint32_t)__builtin_ctzll(m));
    for (uint64_t m = hops; m != 0ull; m &= m - 1ull) a0c += lane_f64(ao, (uint32_t)__builtin_ctzll(m));
    const U4 o = philox10_u(v, kSelfId, c.step, ctr_word3(ri.id, 0u, kCrit, 0u), a.seed_lo, a.seed_hi);
    const double target = uniform01(o.x) * a0c;
    double acc = 0.0;
    int kind = 0, idx = -1, lastkind = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h)
        for (uint64_t m = crit[h] & __ballot(aj[h] > 0.0); m != 0ull && kind == 0; m &= m - 1ull) {
            const uint32_t l = (uint32_t)__builtin_ctzll(m);
            acc += lane_f64(aj[h], l);
            idx = (int)l + 64 * h;
            lastkind = 1;
            if (target < acc) kind = 1;
        }
    for (uint64_t m = hops & __ballot(ao > 0.0); m != 0ull && kind == 0; m &= m - 1ull) {
        const uint32_t l = (uint32_t)__builtin_ctzll(m);
        acc += lane_f64(ao, l);
        idx = (int)l;
        lastkind = 2;
        if (target < acc) kind = 2;
    }
    if (kind == 0) kind = lastkind;
    c.ev_kind = kind;
    c.ev_idx = idx;
    c.ev_dst = kind == 2 ? choose_hop_edge(a, ri, v, row.rb, row.re, row.cw, uniform01(o.y) * W) : v;
}

// ---------------------------------------------------------------------------
// phase A: tau' / tau'' per subvolume, min / argmin per realization
// ---------------------------------------------------------------------------
// Cao's tau' of one subvolume is assembled in three pieces, in this order:
// tau_own (reactions and out-hops), tau_in_edge once per in-neighbour in
// in-CSR order, tau_bound.  The FP64 sums therefore keep one order whether
// the in-edges are walked by the lane itself or staged through LDS.
template <int MS>
struct TauAcc {
    uint32_t x[MS];
    double mu[MS], sig[MS];
    double a0c;
};

template <int MS, int MR>
__device__ __forceinline__ void tau_own(const KernelArgs& a, const NetView& n, const RealInfo& ri, uint32_t v, int c,
                                        TauAcc<MS>& t) {
    const int nc = a.n_critical;
    double av[MR];
    uint32_t crit[(MR + 31) / 32];
    react_props<MR, MS>(n, t.x, c, nc, av, crit);
    const double W = a.wsum[ri.rp_off + v];
    t.a0c = 0.0;
#pragma unroll
    for (int j = 0; j < MR; ++j)
        if (j < n.R && is_crit<MR>(crit, j)) t.a0c += av[j];
#pragma unroll
    for (int s = 0; s < MS; ++s) {
        t.mu[s] = 0.0;
        t.sig[s] = 0.0;
    }
#pragma unroll
    for (int j = 0; j < MR; ++j) {
        if (j >= n.R) break;
        if (is_crit<MR>(crit, j)) continue;
#pragma unroll
        for (int s = 0; s < MS; ++s) {
            if (s >= n.S) break;
            const int nu = n.nu[s * n.R + j];
            if (nu == 0) continue;
            t.mu[s] += (double)nu * av[j];
            t.sig[s] += (double)(nu * nu) * av[j];
        }
    }
#pragma unroll
    for (int s = 0; s < MS; ++s) {
        if (s >= n.S) break;
        const double d = n.d[c * n.S + s];
        if (d > 0.0 && !hop_active(d, t.x[s], nc)) t.a0c += (d * (double)t.x[s]) * W;
        if (hop_active(d, t.x[s], nc)) {
            const double aout = (d * (double)t.x[s]) * W;
            t.mu[s] -= aout;
            t.sig[s] += aout;
        }
    }
}

// In-hops (nu = +1) from one in-neighbour, species whose hops are non-critical:
// du / xu are the neighbour's diffusion constants and counts.  A critical or
// absent hop (count below max(n_c, 1), or d = 0) adds +0 instead of being
// skipped: the sums of the active terms are the same values (only a -0 sum
// would turn into +0, and tau' uses |mu|), without a branch per term.
template <int MS>
__device__ __forceinline__ void tau_in_edge(int S, const double (&du)[MS], const uint32_t (&xu)[MS], double wq,
                                            int nc, TauAcc<MS>& t) {
    const uint32_t nc1 = nc > 1 ? (uint32_t)nc : 1u;
#pragma unroll
    for (int s = 0; s < MS; ++s) {
        // the small instantiations sum every species of the bound (the sums
        // of species S.. are never read; xu and du hold valid padding values
        // for them), so the loop has no runtime exit per species
        if constexpr (MS > 5)
            if (s >= S) break;
        uint32_t xe = xu[s] >= nc1 ? xu[s] : 0u;
        asm("" : "+v"(xe));  // select the count, not its conversion (one select instead of two)
        const double ain = (du[s] * (double)xe) * wq;
        t.mu[s] += ain;
        t.sig[s] += ain;
    }
}

template <int MS>
__device__ __forceinline__ double tau_bound(const KernelArgs& a, const NetView& n, const TauAcc<MS>& t) {
    double tp = kInf;
    const double eps = a.epsilon;
#pragma unroll
    for (int s = 0; s < MS; ++s) {
        if (s >= n.S) break;
        const int hor = n.hor[s];
        if (hor == 0) continue;
        const double mm = fmax(eps_x_over_g(eps, hor, n.mult[s], t.x[s]), 1.0);
        const double t1 = mm / __builtin_fabs(t.mu[s]);
        const double t2 = (mm * mm) / t.sig[s];
        tp = fmin(tp, fmin(t1, t2));
    }
    return tp;
}

// tau' and the critical propensity of one subvolume with counts x, the lane
// walking its own in-edges.
template <int MS, int MR>
__device__ __forceinline__ void tau_subvolume(const KernelArgs& a, const NetView& n, const RealInfo& ri,
                                              const uint32_t* X, const uint32_t (&x)[MS], uint32_t v, double& tp_out,
                                              double& a0c_out) {
    const uint32_t N = ri.N;
    const int c = n.C > 1 ? a.comp[ri.comp_off + v] : 0;
    TauAcc<MS> t;
#pragma unroll
    for (int s = 0; s < MS; ++s) t.x[s] = x[s];
    tau_own<MS, MR>(a, n, ri, v, c, t);
    const bool sym = (ri.flags & 1u) != 0;
    // in-edges: neighbour id and weight in one 8-byte load
    const uint64_t* icw = sym ? a.cw + ri.e_off : a.icw + ri.ie_off;
    const uint32_t* irp = sym ? a.rp + ri.rp_off : a.irp + ri.irp_off;
    const uint32_t ib = irp[v], ie = irp[v + 1];
    // one compartment: the neighbours' diffusion constants are the tile's
    double du[MS];
#pragma unroll
    for (int s = 0; s < MS; ++s) du[s] = n.d[s < n.S ? s : 0];
    if constexpr (MS <= 3) {
        // three in-edges' counts in flight together, the next three's ids and
        // weights behind them (an interior subvolume of a lattice has six): at
        // a few waves per SIMD each trip is one memory round (A-B-C on 24,679
        // subvolumes 8.5 -> 7.8 us against one edge a trip).  One past the
        // row's end adds +0.
        constexpr uint32_t kB = 3;
        uint64_t cw[kB];
#pragma unroll
        for (uint32_t i = 0; i < kB; ++i) cw[i] = ib + i < ie ? icw[ib + i] : (uint64_t)v | kOneW;
        for (uint32_t q = ib; q < ie; q += kB) {
            uint32_t xu[kB][MS];
            uint32_t u[kB];
            double wq[kB];
#pragma unroll
            for (uint32_t i = 0; i < kB; ++i) {
                u[i] = (uint32_t)cw[i];
                wq[i] = (double)__uint_as_float((uint32_t)(cw[i] >> 32));
#pragma unroll
                for (int s = 0; s < MS; ++s) xu[i][s] = X[ri.x_off + (uint64_t)(s < n.S ? s : n.S - 1) * N + u[i]];
            }
#pragma unroll
            for (uint32_t i = 0; i < kB; ++i)
                cw[i] = q + kB + i < ie ? icw[q + kB + i] : (uint64_t)v | kOneW;
            int cu[kB];
#pragma unroll
            for (uint32_t i = 0; i < kB; ++i) cu[i] = n.C > 1 ? a.comp[ri.comp_off + u[i]] : 0;
#pragma unroll
            for (uint32_t i = 0; i < kB; ++i) {
                if (n.C > 1) {
#pragma unroll
                    for (int s = 0; s < MS; ++s) du[s] = n.d[cu[i] * n.S + (s < n.S ? s : 0)];
                }
#pragma unroll
                for (int s = 0; s < MS; ++s) xu[i][s] = q + i < ie ? xu[i][s] : 0u;
                tau_in_edge<MS>(n.S, du, xu[i], wq[i], a.n_critical, t);
            }
        }
        tp_out = tau_bound<MS>(a, n, t);
        a0c_out = t.a0c;
        return;
    }
    // software pipeline: in-edge q's counts were requested in iteration q-1,
    // in-edge q+1's id and weight in iteration q-1 too, so each iteration
    // waits on nothing issued in it
    const uint64_t cw0 = ib < ie ? icw[ib] : (uint64_t)v | kOneW;
    const uint64_t cw1 = ib + 1u < ie ? icw[ib + 1u] : (uint64_t)v | kOneW;
    uint32_t u_cur = (uint32_t)cw0;
    float w_cur = __uint_as_float((uint32_t)(cw0 >> 32));
    uint32_t u_next = (uint32_t)cw1;
    float w_next = __uint_as_float((uint32_t)(cw1 >> 32));
    uint32_t xu[MS];
#pragma unroll
    for (int s = 0; s < MS; ++s) xu[s] = X[ri.x_off + (uint64_t)(s < n.S ? s : n.S - 1) * N + u_cur];
    for (uint32_t q = ib; q < ie; ++q) {
        const uint32_t u = u_cur;
        const double wq = (double)w_cur;
        uint32_t xc[MS];
#pragma unroll
        for (int s = 0; s < MS; ++s) xc[s] = xu[s];
        u_cur = u_next;
        w_cur = w_next;
        if (q + 1u < ie) {
#pragma unroll
            for (int s = 0; s < MS; ++s) xu[s] = X[ri.x_off + (uint64_t)(s < n.S ? s : n.S - 1) * N + u_cur];
            if (q + 2u < ie) {
                const uint64_t cw2 = icw[q + 2u];
                u_next = (uint32_t)cw2;
                w_next = __uint_as_float((uint32_t)(cw2 >> 32));
            }
        }
        if (n.C > 1) {
            const int cu = a.comp[ri.comp_off + u];
#pragma unroll
            for (int s = 0; s < MS; ++s) du[s] = n.d[cu * n.S + (s < n.S ? s : 0)];
        }
        tau_in_edge<MS>(n.S, du, xc, wq, a.n_critical, t);
    }
    tp_out = tau_bound<MS>(a, n, t);
    a0c_out = t.a0c;
}

// Wavefront reductions on DPP lane shifts (row_shr 1, 2, 4, 8, then the two
// row broadcasts; lane 63 ends with all 64): an LDS permute per step and word
// instead takes several times as long, and these sit at the end of every tile.
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t identity, uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)identity, (int)x, CTRL, ROWS, 0xF, false);
}

template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned long long dpp_u64(unsigned long long identity, unsigned long long x) {
    const uint32_t lo = dpp_u32<CTRL, ROWS>((uint32_t)identity, (uint32_t)x);
    const uint32_t hi = dpp_u32<CTRL, ROWS>((uint32_t)(identity >> 32), (uint32_t)(x >> 32));
    return ((unsigned long long)hi << 32) | lo;
}

template <class F>
__device__ __forceinline__ unsigned long long wave_fold_u64(unsigned long long identity, unsigned long long x, F f) {
    x = f(x, dpp_u64<0x111, 0xF>(identity, x));
    x = f(x, dpp_u64<0x112, 0xF>(identity, x));
    x = f(x, dpp_u64<0x114, 0xF>(identity, x));
    x = f(x, dpp_u64<0x118, 0xF>(identity, x));
    x = f(x, dpp_u64<0x142, 0xA>(identity, x));
    x = f(x, dpp_u64<0x143, 0xC>(identity, x));
    return ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(x >> 32), 63) << 32) |
           (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}

template <class F>
__device__ __forceinline__ uint32_t wave_fold_u32(uint32_t identity, uint32_t x, F f) {
    x = f(x, dpp_u32<0x111, 0xF>(identity, x));
    x = f(x, dpp_u32<0x112, 0xF>(identity, x));
    x = f(x, dpp_u32<0x114, 0xF>(identity, x));
    x = f(x, dpp_u32<0x118, 0xF>(identity, x));
    x = f(x, dpp_u32<0x142, 0xA>(identity, x));
    x = f(x, dpp_u32<0x143, 0xC>(identity, x));
    return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}

__device__ __forceinline__ double wave_min(double x) {
    return __longlong_as_double((long long)wave_fold_u64(
        (unsigned long long)__double_as_longlong(kInf), (unsigned long long)__double_as_longlong(x),
        [](unsigned long long p, unsigned long long q) {
            return (unsigned long long)__double_as_longlong(
                fmin(__longlong_as_double((long long)p), __longlong_as_double((long long)q)));
        }));
}

// (tp, t2, v2) <- min tau', argmin tau'' (lowest subvolume on ties) over the
// wavefront, in every lane.  Every lane of the wavefront takes part.
__device__ __forceinline__ void reduce_partA(double& tp, double& t2, uint32_t& v2) {
    tp = wave_min(tp);
    if (__ballot(t2 < kInf) == 0ull) {  // no critical channel: the usual case
        v2 = wave_fold_u32(0xFFFFFFFFu, v2, [](uint32_t p, uint32_t q) { return min(p, q); });
        t2 = kInf;
        return;
    }
    const double m = wave_min(t2);
    v2 = wave_fold_u32(0xFFFFFFFFu, t2 == m ? v2 : 0xFFFFFFFFu, [](uint32_t p, uint32_t q) { return min(p, q); });
    t2 = m;
}

template <int MS, int MR>
__device__ void finalize_A(const KernelArgs& a, const NetView& n, const RealInfo& ri, uint32_t r,
                           double tp, double t2, uint32_t v2, RealCtl c) {
    const bool lead = (threadIdx.x & 63u) == 0u;
    if (tp == kInf && t2 == kInf) {
        c.status = kAbsorbed;
        c.done = 1u;
        if (lead) {
            a.ctl[r] = c;
            atomicAdd(a.ndone, 1u);
        }
        return;
    }
    c.tau_p = tp;
    c.tau2 = t2;
    c.vstar = v2;
    c.learned = (a.learned_on && !c.fallback) ? 1u : 0u;
    c.ev_kind = 0;
    c.ev_idx = -1;
    c.ev_dst = v2;
    decide(c);
    // the event is needed only if tau'' <= tau' (a leap-back halves tau' and
    // can lift the clamp to t_end, but never makes a larger tau'' fire)
    if (t2 < kInf && t2 <= tp) choose_event(a, ri, c, count_buf(a, c.cur));
    if (lead) a.ctl[r] = c;
}

// Cao's tau' / tau'' of one tile's subvolumes into the tile partial (the
// debug outputs, when given, get every subvolume's values instead).
// (tp, t2, v2) <- min tau', argmin tau'' (lowest subvolume on ties) of
// itself and (otp, ot2, ov)
__device__ __forceinline__ void merge_partA(double& tp, double& t2, uint32_t& v2, double otp, double ot2,
                                            uint32_t ov) {
    tp = fmin(tp, otp);
    if (ot2 < t2 || (ot2 == t2 && ov < v2)) {
        t2 = ot2;
        v2 = ov;
    }
}

// Completes the edge-parallel leap at subvolume v of tile t: x and y its counts
// before and after (y mod 2^32), nx the latter in full; their copies go to the
// two buffers left over.  Returns whether a count left its range.
template <int MS>
__device__ __forceinline__ bool finish_counts(const KernelArgs& a, int S, const RealInfo& ri, uint32_t cur,
                                              uint32_t tgt, uint32_t t, uint32_t v, uint32_t (&x)[MS],
                                              uint32_t (&y)[MS], long long (&nx)[MS]) {
    uint32_t z, w;
    spare_bufs(cur, tgt, z, w);
    const uint32_t* X = count_buf(a, cur);
    const uint32_t* Y = count_buf(a, tgt);
    uint32_t *Z = count_buf(a, z), *W = count_buf(a, w);
    const bool wide = wave_uniform(ro(a.wide)[t]) != 0u;
#pragma unroll
    for (int s = 0; s < MS; ++s) {
        const uint64_t at = ri.x_off + (uint64_t)s * ri.N + v;
        x[s] = s < S ? X[at] : 0u;
        y[s] = s < S ? Y[at] : 0u;
    }
    bool out = false;
#pragma unroll
    for (int s = 0; s < MS; ++s) {
        nx[s] = 0;
        if (s >= S) continue;
        const uint64_t at = ri.x_off + (uint64_t)s * ri.N + v;
        long long b = 0;
        if (wide) {
            b = (long long)a.gdelta[at];
            if (b != 0) a.gdelta[at] = 0ull;
        }
        b += (long long)(int32_t)(y[s] - x[s] - (uint32_t)b);
        nx[s] = (long long)x[s] + b;
        out = out || nx[s] < 0 || nx[s] > 0xFFFFFFFFll;
        Z[at] = y[s];
        W[at] = x[s];
    }
    if (wide && (v & 63u) == 0u) a.wide[t] = 0u;  // (a tile's first subvolume: lane 0)
    return out;
}

// spec: the counts the leap pass just wrote (the buffer that becomes current
// if the step is accepted) and the next step's counter; fin: and completes
// the leap on the way.  (A kernel of its own between the two passes read
// counts and 64-bit balances and wrote the new counts: 20 us of the step on
// the 1M-subvolume Brusselator mesh, 4.4 us where the launch was all of it.)
template <int MS, int MR>
__device__ __forceinline__ void cao_tau_tile(const KernelArgs& a, const NetView& n, const RealInfo& ri,
                                             const cptr<RealCtl> cp, const TileEnt& te, uint32_t t, bool dbg,
                                             bool spec = false, bool fin = false) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t cur = wave_uniform(cp->cur), tgt = wave_uniform(cp->tgt);
    const uint32_t* X = count_buf(a, spec ? tgt : cur);
    const uint32_t v = te.v0 + lane;
    double tp = kInf, t2 = kInf, a0c = 0.0;
    uint32_t v2 = v;
    bool out = false;
    if (v < ri.N) {
        uint32_t x[MS];
#pragma unroll
        for (int s = 0; s < MS; ++s) x[s] = s < n.S ? X[ri.x_off + (uint64_t)s * ri.N + v] : 0u;
        tau_subvolume<MS, MR>(a, n, ri, X, x, v, tp, a0c);
        if (a0c > 0.0) {
            const uint32_t step = wave_uniform(cp->step) + (spec ? 1u : 0u);
            const U4 o = philox10_u(v, kSelfId, step, ctr_word3(ri.id, 0u, kTau2, 0u), a.seed_lo, a.seed_hi);
            t2 = -dlog(uniform01(o.x)) / a0c;
        }
        if (dbg) {
            const uint64_t base = ri.x_off / (uint64_t)n.S;
            a.dbg_tp[base + v] = tp;
            a.dbg_a0c[base + v] = a0c;
            a.dbg_t2[base + v] = t2;
        }
    }
    if (dbg) return;
    if (fin && v < ri.N) {  // (at the end: nothing of the sums is live any more)
        uint32_t xo[MS], xn[MS];
        long long nx[MS];
        out = finish_counts<MS>(a, n.S, ri, cur, tgt, t, v, xo, xn, nx);
    }
    if (fin && __ballot(out) != 0ull && lane == 0) a.partB_tile[t].bad |= 1u;
    reduce_partA(tp, t2, v2);
    if (lane == 0) a.partA_tile[t] = PartA{tp, t2, v2, 0u};
}

// The one-compartment tau pass of 3 to 5 species fits in 64 VGPRs without
// spills; asking for 8 waves per SIMD (70 VGPRs and 7 waves otherwise)
// hides more of its gathers' latency (Brusselator mesh 77.6 -> 74.8 us; the
// one-species instantiation measured slower with it, 11.3 -> 12.4 us).
template <int MS, int MR, bool MC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(!MC && MS >= 3 && MS <= 5 ? 8 : 1)))
void phase_a_kernel(KernelArgs a0) {
    for (uint32_t it = 0;; ++it) {
        const uint32_t t = tile_at(it, a0.ntiles, a0.waves_per_block);
        if (t == 0xFFFFFFFFu) break;
        const KernelArgs& a = tile_args();
        const NetView n = net_view<MC>(a);
        const TileEnt te = ld_ro(a.tiles + t);
        const uint32_t r = wave_uniform(te.r);
        const RealInfo ri = ld_ro(a.info + r);
        const cptr<RealCtl> cp = ro(a.ctl + r);
        const uint32_t done = wave_uniform(cp->done), retry = wave_uniform(cp->retry);
        const bool dbg = a.dbg_tp != nullptr;
        // (in the folded order a retried leap has just been made, so only
        // realizations that did not leap are skipped)
        const bool spec = a.tau_spec != 0u && !dbg;
        if (!dbg && (done || (retry && !spec))) continue;
        cao_tau_tile<MS, MR>(a, n, ri, cp, te, t, dbg, spec, spec && a.finish_in_tau);
    }
}

// One block per realization: min tau' / argmin tau'' over the realization's
// tile partials (written by phase A; the kernel boundary makes them visible),
// then the step decision.
// Threads of decide_kernel and commit_decide_kernel: 4 wavefronts.  With
// 1,024 tile partials per chunk block that is 4 loads per thread, one
// round; 16-wavefront blocks, one load per thread, measured slower (the
// barrier and the 16-way reduction outweigh the round they save:
// commit_decide_kernel 12.8 -> 9.8 us on the Brusselator mesh).
template <int MS>
constexpr uint32_t decide_threads() { return 256u; }

// decide_kernel runs decide_chunks blocks per realization (one per 1,024
// tile partials of the largest realization, at most kDecideChunks): each
// reduces one chunk of the realization's tile partials (the reads spread
// over as many CUs), publishes its partial and counts itself in; the last
// block of the realization reduces the chunk partials and decides the
// step.  Release fence before the count, acquire fence after it (agent
// scope: the blocks run on different XCDs); the last block clears the
// counter for the next step (the next launch is ordered after this
// kernel).  With one block per realization it decides directly.
template <int MS>
__device__ __forceinline__ void reduce_block_partA(double& tp, double& t2, uint32_t& v2, double* s_tp, double* s_t2,
                                                   uint32_t* s_v2) {
    reduce_partA(tp, t2, v2);
    const uint32_t wv = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    if (lane == 0) {
        s_tp[wv] = tp;
        s_t2[wv] = t2;
        s_v2[wv] = v2;
    }
    __syncthreads();
    if (wv == 0) {  // the first wavefront, every lane alike
        for (uint32_t w = 1; w < (blockDim.x >> 6); ++w) {
            tp = fmin(tp, s_tp[w]);
            if (s_t2[w] < t2 || (s_t2[w] == t2 && s_v2[w] < v2)) {
                t2 = s_t2[w];
                v2 = s_v2[w];
            }
        }
    }
}

template <int MS, int MR>
__global__ __launch_bounds__(decide_threads<MS>()) void decide_kernel(KernelArgs a) {
    const uint32_t nch = a.decide_chunks;
    const uint32_t r = blockIdx.x / nch, chunk = blockIdx.x % nch;
    if (r >= a.nreal) return;
    // the realization's control block and info in one round of loads
    const RealInfo ri = ld_ro(a.info + r);
    const RealCtl c0 = ld_ro(a.ctl + r);
    if (c0.done || c0.retry) return;  // the same in every block of the realization
    __shared__ double s_tp[16], s_t2[16];
    __shared__ uint32_t s_v2[16];
    __shared__ uint32_t s_last;
    const uint32_t per = (ri.ntiles + nch - 1u) / nch;
    const uint32_t qb = min(chunk * per, ri.ntiles), qe = min(qb + per, ri.ntiles);
    double tp = kInf, t2 = kInf;
    uint32_t v2 = 0xFFFFFFFFu;
    // 8 independent loads in flight per thread
    for (uint32_t q0 = qb; q0 < qe; q0 += 8u * blockDim.x) {
        PartA p[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t q = q0 + (uint32_t)i * blockDim.x + threadIdx.x;
            p[i] = q < qe ? a.partA_tile[ri.tile_begin + q] : PartA{kInf, kInf, 0xFFFFFFFFu, 0u};
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            tp = fmin(tp, p[i].tp);
            if (p[i].t2 < t2 || (p[i].t2 == t2 && p[i].v2 < v2)) {
                t2 = p[i].t2;
                v2 = p[i].v2;
            }
        }
    }
    reduce_block_partA<MS>(tp, t2, v2, s_tp, s_t2, s_v2);
    if (nch == 1u) {
        if (threadIdx.x < 64u) finalize_A<MS, MR>(a, net_view(a), ri, r, tp, t2, v2, c0);
        return;
    }
    if (threadIdx.x == 0) {
        a.partA_chunk[r * nch + chunk] = PartA{tp, t2, v2, 0u};
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        s_last = atomicAdd(&a.decide_cnt[r], 1u) == nch - 1u ? 1u : 0u;
    }
    __syncthreads();
    if (!s_last || threadIdx.x >= 64u) return;
    // the last block of the realization: its first wavefront decides
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    const uint32_t lane = threadIdx.x;
    PartA p{kInf, kInf, 0xFFFFFFFFu, 0u};
    if (lane < nch) p = a.partA_chunk[r * nch + lane];
    tp = p.tp;
    t2 = p.t2;
    v2 = p.v2;
    reduce_partA(tp, t2, v2);
    if (lane == 0) a.decide_cnt[r] = 0u;
    finalize_A<MS, MR>(a, net_view(a), ri, r, tp, t2, v2, c0);
}

// ---------------------------------------------------------------------------
// phase B: leap + critical event + negative check, commit / leap-back
// ---------------------------------------------------------------------------
struct StepView {
    double tau;
    uint32_t step, attempt, real;
    int crit, ev_kind, ev_idx;
    uint32_t vstar, ev_dst;
};

template <int MS, int MR>
__device__ __forceinline__ bool leap_subvolume(const KernelArgs& a, const NetView& n, const RealInfo& ri,
                                               const uint32_t* X, uint32_t* Xn, uint32_t v,
                                               const StepView& sv, unsigned long long& fire_out,
                                               uint32_t& viol) {
    const uint32_t N = ri.N;
    const int nc = a.n_critical;
    uint32_t x[MS];
#pragma unroll
    for (int s = 0; s < MS; ++s) x[s] = s < n.S ? X[ri.x_off + (uint64_t)s * N + v] : 0u;
    const int c = n.C > 1 ? a.comp[ri.comp_off + v] : 0;
    double av[MR];
    uint32_t crit[(MR + 31) / 32];
    react_props<MR, MS>(n, x, c, nc, av, crit);
    long long nx[MS];
#pragma unroll
    for (int s = 0; s < MS; ++s) nx[s] = (long long)x[s];
    unsigned long long fire = 0;
    const double tau = sv.tau;
    const uint32_t k0 = a.seed_lo, k1 = a.seed_hi;

    // non-critical reactions: k_j ~ Poisson(tau a_j)
    {
        uint32_t blk = 0xFFFFFFFFu;
        U4 o{0, 0, 0, 0};
        const uint32_t c3base = ctr_word3(sv.real, sv.attempt, kReact, 0u);
        for (int j = 0; j < n.R; ++j) {
            if (is_crit<MR>(crit, j) || !(av[j] > 0.0)) continue;
            const uint32_t b = (uint32_t)j >> 4;
            if (b != blk) {
                o = philox10_u(v, kSelfId, sv.step, c3base | b, k0, k1);
                blk = b;
            }
            const long long k = leap_draw(tau * av[j], coarse_byte(o, (uint32_t)j), v, kSelfId, sv.step, c3base,
                                          k0, k1, (uint32_t)j);
            fire += (unsigned long long)k;
#pragma unroll
            for (int s = 0; s < MS; ++s)
                if (s < n.S) nx[s] += k * (long long)n.nu[s * n.R + j];
        }
    }

    const bool weighted = (ri.flags & 2u) != 0;
    const bool sym = (ri.flags & 1u) != 0;
    const uint32_t rb = a.rp[ri.rp_off + v], re = a.rp[ri.rp_off + v + 1];
    double dx[MS];
    bool act[MS];
#pragma unroll
    for (int s = 0; s < MS; ++s) {
        const double d = s < n.S ? n.d[c * n.S + s] : 0.0;
        act[s] = s < n.S && hop_active(d, x[s], nc);
        dx[s] = d * (double)x[s];
    }
    const uint32_t c3hop = ctr_word3(sv.real, sv.attempt, kHop, 0u);
    if (sym) {
        // One coarse block per (edge, species pair) serves both directions of
        // both species.  Pairs outer (unrolled: static indices keep the count
        // accumulators in registers), edges inner (rolled: few live values).
        const uint32_t* colp = a.col + ri.e_off;
        const float* wp = a.w + ri.e_off;
#pragma unroll
        for (int s0 = 0; s0 < MS; s0 += 2) {
            if (s0 >= n.S) break;
            const bool two = s0 + 1 < MS && s0 + 1 < n.S;
            const bool act0 = act[s0], act1 = two && act[s0 + 1 < MS ? s0 + 1 : s0];
            const double dx0 = dx[s0], dx1 = two ? dx[s0 + 1 < MS ? s0 + 1 : s0] : 0.0;
            const uint32_t* X0 = X + ri.x_off + (uint64_t)s0 * N;
            const uint32_t* X1 = two ? X0 + N : X0;
            const uint32_t cb = c3hop | ((uint32_t)s0 >> 3);
            const uint32_t w0 = 2u * (uint32_t)s0;
            long long d0 = 0, d1 = 0;
            for (uint32_t q = rb; q < re; ++q) {
                const uint32_t u = colp[q];
                const double wq = weighted ? (double)wp[q] : 1.0;
                const int cu = n.C > 1 ? a.comp[ri.comp_off + u] : 0;
                const uint32_t xu0 = X0[u];
                const uint32_t xu1 = two ? X1[u] : 0u;
                const double du0 = n.d[cu * n.S + s0];
                const double du1 = two ? n.d[cu * n.S + s0 + 1] : 0.0;
                const double lo0 = act0 ? tau * (dx0 * wq) : 0.0;
                const double lo1 = act1 ? tau * (dx1 * wq) : 0.0;
                const double li0 = hop_active(du0, xu0, nc) ? tau * ((du0 * (double)xu0) * wq) : 0.0;
                const double li1 = (two && hop_active(du1, xu1, nc)) ? tau * ((du1 * (double)xu1) * wq) : 0.0;
                if (!(lo0 > 0.0 || lo1 > 0.0 || li0 > 0.0 || li1 > 0.0)) continue;
                const uint32_t lo = v < u ? v : u, hi = v < u ? u : v;
                const uint32_t dout = v > u ? 1u : 0u, din = 1u - dout;
                const U4 o = philox10_u(lo, hi, sv.step, cb, k0, k1);
                auto hop = [&](double l, uint32_t w) {
                    return leap_draw(l, coarse_byte(o, w), lo, hi, sv.step, c3hop, k0, k1, w);
                };
                if (lo0 > 0.0) {
                    const long long k = hop(lo0, w0 + dout);
                    d0 -= k;
                    fire += (unsigned long long)k;
                }
                if (li0 > 0.0) d0 += hop(li0, w0 + din);
                if (lo1 > 0.0) {
                    const long long k = hop(lo1, w0 + 2u + dout);
                    d1 -= k;
                    fire += (unsigned long long)k;
                }
                if (li1 > 0.0) d1 += hop(li1, w0 + 2u + din);
            }
#pragma unroll
            for (int q = 0; q < MS; ++q) {
                if (q == s0) nx[q] += d0;
                if (q == s0 + 1) nx[q] += d1;
            }
        }
    } else {
        for (uint32_t q = rb; q < re; ++q) {
            const uint32_t u = a.col[ri.e_off + q];
            const double wq = weighted ? (double)a.w[ri.e_off + q] : 1.0;
            const uint32_t lo = v < u ? v : u, hi = v < u ? u : v;
            const uint32_t dout = v > u ? 1u : 0u;
#pragma unroll
            for (int s = 0; s < MS; ++s) {
                if (s >= n.S) break;
                if (!act[s]) continue;
                const uint32_t wd = 2u * (uint32_t)s + dout;
                const U4 o = philox10_u(lo, hi, sv.step, c3hop | (wd >> 4), k0, k1);
                const long long k =
                    leap_draw(tau * (dx[s] * wq), coarse_byte(o, wd), lo, hi, sv.step, c3hop, k0, k1, wd);
                nx[s] -= k;
                fire += (unsigned long long)k;
            }
        }
        const uint32_t ib = a.irp[ri.irp_off + v], ie = a.irp[ri.irp_off + v + 1];
        for (uint32_t q = ib; q < ie; ++q) {
            const uint32_t u = a.icol[ri.ie_off + q];
            const double wq = weighted ? (double)a.iw[ri.ie_off + q] : 1.0;
            const int cu = n.C > 1 ? a.comp[ri.comp_off + u] : 0;
            const uint32_t lo = v < u ? v : u, hi = v < u ? u : v;
            const uint32_t din = u > v ? 1u : 0u;
#pragma unroll
            for (int s = 0; s < MS; ++s) {
                if (s >= n.S) break;
                const uint32_t xu = X[ri.x_off + (uint64_t)s * N + u];
                const double du = n.d[cu * n.S + s];
                if (!hop_active(du, xu, nc)) continue;
                const uint32_t wd = 2u * (uint32_t)s + din;
                const U4 o = philox10_u(lo, hi, sv.step, c3hop | (wd >> 4), k0, k1);
                nx[s] += leap_draw(tau * ((du * (double)xu) * wq), coarse_byte(o, wd), lo, hi, sv.step, c3hop, k0,
                                   k1, wd);
            }
        }
    }

    // the critical event (one per global step, in the argmin-tau'' subvolume)
    if (sv.crit) {
        if (v == sv.vstar) {
            if (sv.ev_kind == 1) {
#pragma unroll
                for (int s = 0; s < MS; ++s)
                    if (s < n.S) nx[s] += n.nu[s * n.R + sv.ev_idx];
                fire += 1ull;
            } else if (sv.ev_kind == 2) {
#pragma unroll
                for (int s = 0; s < MS; ++s)
                    if (s == sv.ev_idx) nx[s] -= 1;
                fire += 1ull;
            }
        }
        if (sv.ev_kind == 2 && v == sv.ev_dst && sv.ev_dst != sv.vstar) {
#pragma unroll
            for (int s = 0; s < MS; ++s)
                if (s == sv.ev_idx) nx[s] += 1;
        }
    }
    bool bad = false;
#pragma unroll
    for (int s = 0; s < MS; ++s) {
        if (s >= n.S) break;
        bad = bad || nx[s] < 0 || nx[s] > 0xFFFFFFFFll;
        Xn[ri.x_off + (uint64_t)s * N + v] = (uint32_t)nx[s];
    }
    fire_out = fire;
    viol = a.judge_on ? leap_condition_broken<MS, MR>(n, c, nc, a.epsilon, a.theta, x, nx, av, crit) : 0u;
    return bad;
}

// ---------------------------------------------------------------------------
// Edge-parallel leap of one tile.
//
// Each pair of linked subvolumes {v, u}, v < u, is drawn once, by the tile of
// its lower end: the tile's forward-CSR entries are contiguous, lane l takes
// entries l, l+64, ... (coalesced loads, no divergence from uneven degrees),
// each one 8-byte word that holds the neighbour, the owning subvolume's
// index in the tile and the weight (an asymmetric topology's weight of the
// hop back in a second array), and draws both hop directions of every species
// from the pair's coarse Philox block; then lane i draws the reactions of
// subvolume v0+i (one coarse block per 16 reactions).
// Balances of the tile's own subvolumes collect in LDS, those of other
// tiles' subvolumes go straight to the target buffer, which holds a copy of
// the counts; integer atomics keep every sum exact and order-free.  The next
// pass completes the leap (finish_counts) once every draw is in.
//
// Compacted draws.  Almost every draw of a step is 0 where hop means are
// small (~1e-3 on the headline mesh), so the walk only applies the zero
// shortcut to the coarse byte of each draw's word: a draw it cannot settle
// as 0 goes to the wavefront's LDS queue as its code and coarse byte, and the
// whole wavefront draws the queued ones, one per lane -- the fine bits, the
// float squeeze, then the double search where the squeeze cannot decide, PTRS
// for a mean of 10 or more -- so the fine block and the search run once per 64
// open draws instead of once per draw site.  The queue is drawn when the next
// 64 entries' open draws might not fit and at the end of the walk; a drained
// walk forms its loads again, so nothing of it is live across the sampler.
// Every draw is inline: no call keeps the kernel at the walk's registers.
// (A tile whose queue overflowed, or that held a mean of 10 or more, used to
// go to a second kernel that drew one draw site at a time on two blocks per
// CU: where means are ~0.5, as in the bistable model at equilibrium, every
// tile did, 80 us of a 127 us step on the 64^3 grid; and where none did, its
// empty launch took 4.4 us.)
// ---------------------------------------------------------------------------
// A tile counts as beyond its queue (plis_redo_tiles) with more open draws
// than kQueue or a mean that may be 10 or more: a hop's float mean is within
// 8 * 2^-24 (relative) of its double mean, so one at or below kPtrsMaybeF is
// a double mean below 10.
constexpr uint32_t kQueue = 256;
constexpr float kPtrsMaybeF = 9.9999f;
constexpr uint32_t kQueueReact = 0x80000000u;  // reaction: flag | lane << 16 | j << 8 | byte
                                               // hop: entry << 12 | w << 8 | byte (kMaxTileEdges)
// Draws that are made at once instead of queued: from kInlineDraws open ones
// per species among 64 entries, or of one reaction in a tile, on, one fine block
// and one squeeze per direction for all 64 lanes cost less than each queued
// draw's own block, entry and counts (bistable 64^3 grid at its equilibrium
// 38 -> 30 us a leap with thresholds of 32 or 48, 30.1 with 16).  Means of kInlineMaxF or more and draws
// the squeeze leaves open are queued all the same.  Networks of more than 3
// species have no registers left for it.
constexpr uint32_t kInlineDraws = 32;
constexpr float kInlineMaxF = 9.99f;
constexpr float kNoHop = -0x1p+100f;           // rate of a hop that is critical or absent: never open

// One wavefront's staging.  The queue takes all draws of 64 entries.
template <int MS, bool GEN>
struct LeapLds {
    static constexpr uint32_t kCap = MS > 2 ? 128u * MS : 256u;
    uint32_t x[MS][kTile];   // the tile's counts
    float rate[MS][kTile];   // their hops' coarse rates (kCoarseScale tau d x; kNoHop)
    int32_t del[MS][kTile];  // the tile's balances
    uint32_t q[kCap];
    int32_t c[GEN ? kTile : 1];
    // what each wavefront of a split tile found: {firings, open draws, a mean
    // of 10 or more}
    unsigned long long part_fire;
    uint32_t part_opened, part_big;
};

// A wavefront's share of a tile: wavefront `part` of `parts` (1, or the block's
// 4) takes every parts-th group of 64 entries, reaction and species.
template <uint32_t PARTS>
struct TileShare {
    static constexpr uint32_t parts = PARTS;
    uint32_t part;
    __device__ __forceinline__ void sync() const {
        if (parts > 1u) __syncthreads();
        else lds_wave_sync();
    }
};

__device__ __forceinline__ uint64_t wave_ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }

__device__ __forceinline__ uint32_t lanes_below(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

__device__ __forceinline__ double hop_mean(double d, uint32_t x, double wq, double tau, int nc) {
    return hop_active(d, x, nc) ? tau * ((d * (double)x) * wq) : 0.0;
}

// The same mean in single precision for the fast path: tau, d and x rounded
// to float (w already is), three float products; within 8 2^-24 of it.
__device__ __forceinline__ float hop_mean_f(double d, uint32_t x, float w, float tauf, int nc) {
    return hop_active(d, x, nc) ? tauf * (((float)d * (float)x) * w) : 0.0f;
}

// Balance b of species s at subvolume u: through LDS in the tile, else
// straight to the target buffer Y (see KernelArgs::gdelta for a wide one).
template <int MS, bool GEN>
__device__ __forceinline__ void add_balance(const KernelArgs& a, const RealInfo& ri, LeapLds<MS, GEN>& L, uint32_t* Y,
                                            uint32_t v0, int s, uint32_t u, long long b) {
    const uint64_t at = ri.x_off + (uint64_t)s * ri.N + u;
    if (b <= -(long long)a.narrow || b >= (long long)a.narrow) {
        atomicAdd(&a.gdelta[at], (unsigned long long)b);
        atomicOr(&a.wide[ri.tile_begin + u / (uint32_t)kTile], 1u);
        atomicAdd(&Y[at], (uint32_t)b);
    } else if (u - v0 < (uint32_t)kTile) {
        atomicAdd(&L.del[s][u - v0], (int32_t)b);
    } else {
        atomicAdd(&Y[at], (uint32_t)b);
    }
}

// One queued draw: its fine bits complete the word the walk queued the
// coarse byte of (one Philox call, whichever the kind), then the sampler,
// applied to the balances.  big: the mean may be 10 or more.
template <int MS, bool GEN>
__device__ __forceinline__ void drain_draw(const KernelArgs& a, const NetView& n, const RealInfo& ri,
                                           const uint32_t* X, uint32_t* Y, uint32_t v0, const StepView& sv,
                                           LeapLds<MS, GEN>& L, uint32_t eb, uint32_t code, unsigned long long& fire, bool& big) {
    const bool react = (code & kQueueReact) != 0u;
    const uint32_t hb = code & 255u;
    uint32_t i, c1, w, c3;
    bool fwd = true;
    float lf;
    double lam;
    if (react) {
        i = (code >> 16) & 63u;
        w = (code >> 8) & 255u;
        double aj = n.k[(n.C > 1 ? L.c[GEN ? i : 0] : 0) * n.R + (int)w];
        const int nr = n.nrs[w];
        for (int r = 0; r < nr; ++r) aj = aj * binom_d(L.x[n.rs[w * 3 + r]][i], n.rr[w * 3 + r]);
        lam = sv.tau * aj;
        lf = (float)lam;
        c1 = kSelfId;
        c3 = ctr_word3(sv.real, sv.attempt, kReact, kFineBlock + (w >> 2));
        big = big || !(lam < kPoissonInvMax);
    } else {
        const uint64_t e = ri.fe_off + eb + (code >> 12);
        const uint64_t cw = a.fcw[e];
        w = (code >> 8) & 15u;
        i = (uint32_t)cw >> 26;
        c1 = (uint32_t)cw & kFwdIdMask;
        fwd = (w & 1u) == 0u;
        const int s = (int)(w >> 1);
        float wf = __uint_as_float((uint32_t)(cw >> 32));
        if constexpr (GEN)
            if (!fwd && a.frw) wf = a.frw[e];
        double d;
        uint32_t xs;
        const bool local = c1 - v0 < (uint32_t)kTile;
        if (fwd) {
            d = n.d[(n.C > 1 ? L.c[GEN ? i : 0] : 0) * n.S + s];
            xs = L.x[s][i];
        } else {
            const int cu = n.C > 1 ? (local ? L.c[GEN ? c1 - v0 : 0] : a.comp[ri.comp_off + c1]) : 0;
            d = n.d[cu * n.S + s];
            xs = local ? L.x[s][c1 - v0] : X[ri.x_off + (uint64_t)s * ri.N + c1];
        }
        lam = hop_mean(d, xs, (double)wf, sv.tau, a.n_critical);
        lf = hop_mean_f(d, xs, wf, (float)sv.tau, a.n_critical);
        c3 = ctr_word3(sv.real, sv.attempt, kHop, kFineBlock + (w >> 2));
        big = big || lf > kPtrsMaybeF;
    }
    const uint32_t word = draw_word(hb, philox10_u(v0 + i, c1, sv.step, c3, a.seed_lo, a.seed_hi), w);
    long long k = lf < kSqueezeMaxF ? poisson_squeeze(lf, __uint2float_rn(word) * 0x1p-32f) : -1;
    if (k < 0) {
        if (lam < kPoissonInvMax) k = inversion_search(lam, word);
        else k = ptrs_draw(lam, DrawId{v0 + i, c1, sv.step, c3, a.seed_lo, a.seed_hi, w & 3u});
    }
    if (k == 0) return;
    fire += (unsigned long long)k;
    if (react) {
        for (int s = 0; s < n.S; ++s) {
            const int nu = n.nu[s * n.R + (int)w];
            if (nu != 0) add_balance(a, ri, L, Y, v0, s, v0 + i, k * (long long)nu);
        }
    } else {
        const int s = (int)(w >> 1);
        const long long b = fwd ? -k : k;  // balance of v0 + i
        add_balance(a, ri, L, Y, v0, s, v0 + i, b);
        add_balance(a, ri, L, Y, v0, s, c1, -b);
    }
}

// The draws of one tile, and the critical event if it is the tile's, into the
// target buffer Y.  Control flow stays
// wave-uniform around every queue append: the loops run the same trip count
// on every lane, lanes without work carry flags.  q_: the wavefront's queue.
// Returns whether some mean was 10 or more, in opened_out the open draws.  GEN: several compartments or an asymmetric
// topology.
template <int MS, int MR, bool GEN, uint32_t PARTS>
__device__ __forceinline__ bool leap_tile_draws(const KernelArgs& a, const NetView& n, const RealInfo& ri,
                                                const uint32_t* X, uint32_t* Y, uint32_t v0, const StepView& sv,
                                                LeapLds<MS, GEN>& L, uint32_t* q_, const TileShare<PARTS>& sh,
                                                unsigned long long& fire, uint32_t& opened_out) {
    static_assert(MS <= 8 && MR <= 16, "one coarse block per pair and per subvolume; hop codes hold w in 4 bits");
    constexpr uint32_t kCap = LeapLds<MS, GEN>::kCap;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t N = ri.N;
    const uint32_t v = v0 + lane;
    const bool vok = v < N;
    const int nc = a.n_critical;
    const uint32_t nc1 = nc > 1 ? (uint32_t)nc : 1u;
    const double tau = sv.tau;
    const uint32_t k0 = a.seed_lo, k1 = a.seed_hi;
    const float scale = (float)tau * kCoarseScale;
    const int cl = (GEN && n.C > 1 && vok) ? a.comp[ri.comp_off + v] : 0;
    float dt[MS];    // one compartment: the species' rate per molecule
    bool dpos[MS];
#pragma unroll
    for (int s = 0; s < MS; ++s) {
        const double d = n.d[s < n.S ? s : 0];
        dt[s] = (float)d * scale;
        dpos[s] = s < n.S && d > 0.0;
        if (sh.parts > 1u && ((uint32_t)s & 3u) != sh.part) continue;
        const uint32_t x = (vok && s < n.S) ? X[ri.x_off + (uint64_t)s * N + v] : 0u;
        L.x[s][lane] = x;
        L.del[s][lane] = 0;
        if (GEN && n.C > 1) {
            const double dc = n.d[cl * n.S + (s < n.S ? s : 0)];
            L.rate[s][lane] = (s < n.S && dc > 0.0 && x >= nc1) ? ((float)dc * scale) * (float)x : kNoHop;
        } else {
            L.rate[s][lane] = (dpos[s] && x >= nc1) ? dt[s] * (float)x : kNoHop;
        }
    }
    if constexpr (GEN) L.c[lane] = cl;
    const uint32_t eb = wave_uniform(a.frp[ri.rp_off + v0]);
    const uint32_t ee = wave_uniform(a.frp[ri.rp_off + min(v0 + (uint32_t)kTile, N)]);
    sh.sync();
    const uint64_t* cwp = a.fcw + ri.fe_off;  // neighbour, row in the tile and weight in one load
    const float* rwp = GEN && a.frw ? a.frw + ri.fe_off : nullptr;
    const uint32_t c3hop = ctr_word3(sv.real, sv.attempt, kHop, 0u);
    const uint32_t c3react = ctr_word3(sv.real, sv.attempt, kReact, 0u);
    const uint32_t nit = (ee - eb + (uint32_t)kTile - 1u) / (uint32_t)kTile;
    uint32_t qn = 0u, opened = 0u;
    bool big = false;
    // software pipeline: an entry's neighbour counts are requested one
    // iteration ahead, its neighbour id and weight two iterations ahead
    // (counts of a neighbour inside the tile are read from global memory
    // too: the staged copy holds the same values)
    auto counts = [&](uint32_t u, uint32_t (&xo)[MS]) {
#pragma unroll
        for (int s = 0; s < MS; ++s) xo[s] = X[ri.x_off + (uint64_t)(s < n.S ? s : n.S - 1) * N + u];
    };
    const uint32_t step64 = sh.parts * (uint32_t)kTile;
    uint32_t it = sh.part;
    int j = (int)(sh.parts - 1u - sh.part);  // (the wavefronts with fewer entries have more reactions)
    for (bool all = false; !all;) {
        if (it < nit) {
            uint32_t e = eb + it * (uint32_t)kTile + lane;
            const uint64_t none = (uint64_t)v0 | kOneW;
            uint64_t cw = e < ee ? cwp[e] : none, cw_next = e + step64 < ee ? cwp[e + step64] : none;
            uint32_t xn[MS];
            counts((uint32_t)cw & kFwdIdMask, xn);
            for (; it < nit; it += sh.parts, e += step64) {
                const bool valid = e < ee;
                const uint32_t i = (uint32_t)cw >> 26;            // the entry's row in the tile
                const uint32_t u = (uint32_t)cw & kFwdIdMask;     // u > v0 + i
                const float w0 = __uint_as_float((uint32_t)(cw >> 32));
                float w1 = w0;
                if constexpr (GEN)
                    if (rwp && valid) w1 = rwp[e];
                uint32_t xc[MS];
#pragma unroll
                for (int s = 0; s < MS; ++s) xc[s] = xn[s];
                cw = cw_next;
                if (e + step64 < ee) {
                    counts((uint32_t)cw & kFwdIdMask, xn);
                    if (e + 2u * step64 < ee) cw_next = cwp[e + 2u * step64];
                }
                int cu = 0;
                if (GEN && n.C > 1 && valid)
                    cu = u - v0 < (uint32_t)kTile ? L.c[GEN ? u - v0 : 0] : a.comp[ri.comp_off + u];
                // rates of the draws w = 2s + direction (0: v0 + i -> u)
                float rate[2 * MS];
                bool any = false;
#pragma unroll
                for (int s = 0; s < MS; ++s) {
                    rate[2 * s] = L.rate[s][i];
                    bool on = xc[s] >= nc1;
                    float r;
                    if (GEN && n.C > 1) {
                        const double d = n.d[cu * n.S + (s < n.S ? s : 0)];
                        on = on && s < n.S && d > 0.0;
                        r = ((float)d * scale) * (float)xc[s];
                    } else {
                        on = on && dpos[s];
                        r = dt[s] * (float)xc[s];
                    }
                    rate[2 * s + 1] = on ? r : kNoHop;
                    any = any || on || rate[2 * s] > 0.0f;
                }
                if (wave_ballot(any && valid) == 0ull) continue;
                const U4 o = philox10_u(v0 + i, u, sv.step, c3hop, k0, k1);
                bool open[2 * MS];
                uint32_t total = 0u;
#pragma unroll
                for (int w = 0; w < 2 * MS; ++w) {
                    open[w] = valid && __builtin_fmaf(rate[w], (w & 1) ? w1 : w0, (float)coarse_byte(o, (uint32_t)w)) > kCoarseTop;
                    total += (uint32_t)__popcll(wave_ballot(open[w]));
                }
                if (qn + total > kCap) break;  // drawn below, then this entry again
                opened += total;
                if constexpr (MS <= 3) {
                    if (total >= kInlineDraws * MS) {
                        U4 f{};
#pragma unroll
                        for (int s = 0; s < MS; ++s) {
                            if (s % 2 == 0)
                                f = philox10_u(v0 + i, u, sv.step, c3hop | (kFineBlock + (uint32_t)s / 2u), k0, k1);
                            int k[2] = {0, 0};
#pragma unroll
                            for (int dir = 0; dir < 2; ++dir) {
                                const int w = 2 * s + dir;
                                // (within 9 2^-24 of the double mean, one rounding more than hop_mean_f)
                                const float lf = (rate[w] * (dir ? w1 : w0)) * (1.0f / kCoarseScale);
                                if (!(open[w] && lf < kInlineMaxF)) continue;
                                const uint32_t word = draw_word(coarse_byte(o, (uint32_t)w), f, (uint32_t)w);
                                const int kd = poisson_squeeze(lf, __uint2float_rn(word) * 0x1p-32f);
                                if (kd < 0) continue;
                                open[w] = false;
                                k[dir] = kd;
                            }
                            fire += (unsigned long long)(uint32_t)(k[0] + k[1]);
                            const int b = k[1] - k[0];  // never wide: a squeezed draw is at most kSqueezeK
                            if (b != 0) {
                                atomicAdd(&L.del[s][i], b);
                                if (u - v0 < (uint32_t)kTile) atomicAdd(&L.del[s][u - v0], -b);
                                else atomicAdd(&Y[ri.x_off + (uint64_t)s * N + u], (uint32_t)-b);
                            }
                        }
                    }
                }
                const uint32_t code = (e - eb) << 12;
#pragma unroll
                for (int w = 0; w < 2 * MS; ++w) {
                    const uint64_t m = wave_ballot(open[w]);
                    if (m == 0ull) continue;
                    if (open[w]) q_[qn + lanes_below(m)] = code | ((uint32_t)w << 8) | coarse_byte(o, (uint32_t)w);
                    qn += (uint32_t)__popcll(m);
                }
            }
        }
        if (it >= nit) {
            // reactions of subvolume v, propensities and criticality as react_props
            // computes them (same operations, one reaction at a time)
            const U4 o = philox10_u(v, kSelfId, sv.step, c3react, k0, k1);
            U4 f{};
            int fine = -1;  // f: the fine bits of reactions 4 fine .. 4 fine + 3
            for (; j < n.R; j += (int)sh.parts) {
                double aj = n.k[cl * n.R + j];
                bool low = false;
                const int nr = n.nrs[j];
                for (int q = 0; q < nr; ++q) {
                    const int sq = n.rs[j * 3 + q], rq = n.rr[j * 3 + q];
                    const uint32_t xs = L.x[sq][lane];
                    aj = aj * binom_d(xs, rq);
                    low = low || below_nc(xs, rq, nc);
                }
                const uint32_t hb = coarse_byte(o, (uint32_t)j);
                bool open = vok && !(n.order[j] > 0 && low) && aj > 0.0 && !coarse_zero(tau * aj, hb);
                uint64_t m = wave_ballot(open);
                uint32_t cnt = (uint32_t)__popcll(m);
                if (qn + cnt > kCap) break;
                opened += cnt;
                if constexpr (MS <= 3) {
                    if (cnt >= kInlineDraws) {
                        if (fine != (j >> 2)) {
                            fine = j >> 2;
                            f = philox10_u(v, kSelfId, sv.step, c3react | (kFineBlock + (uint32_t)fine), k0, k1);
                        }
                        const float lf = (float)(tau * aj);
                        if (open && lf < kInlineMaxF) {
                            const int k = poisson_squeeze(lf, __uint2float_rn(draw_word(hb, f, (uint32_t)j)) * 0x1p-32f);
                            open = k < 0;
                            if (k > 0) {
                                fire += (unsigned long long)(uint32_t)k;
                                for (int s = 0; s < n.S; ++s) {
                                    const int nu = n.nu[s * n.R + j];
                                    if (nu != 0) add_balance(a, ri, L, Y, v0, s, v, (long long)k * (long long)nu);
                                }
                            }
                        }
                        m = wave_ballot(open);
                        cnt = (uint32_t)__popcll(m);
                    }
                }
                if (open) q_[qn + lanes_below(m)] = kQueueReact | (lane << 16) | ((uint32_t)j << 8) | hb;
                qn += cnt;
            }
            all = j >= n.R;
        }
        lds_wave_sync();
        for (uint32_t q = lane; q < qn; q += (uint32_t)kTile)
            drain_draw<MS, GEN>(a, n, ri, X, Y, v0, sv, L, eb, q_[q], fire, big);
        lds_wave_sync();
        qn = 0u;
    }
    if (sv.crit && sh.part == 0u && sv.vstar - v0 < (uint32_t)kTile) {
        if (v == sv.vstar && (sv.ev_kind == 1 || sv.ev_kind == 2)) {
            fire += 1ull;
            if (sv.ev_kind == 1) {
                for (int s = 0; s < n.S; ++s)
                    add_balance(a, ri, L, Y, v0, s, v, (long long)n.nu[s * n.R + sv.ev_idx]);
            } else {
                add_balance(a, ri, L, Y, v0, sv.ev_idx, v, -1ll);
                if (sv.ev_dst != v) add_balance(a, ri, L, Y, v0, sv.ev_idx, sv.ev_dst, 1ll);
            }
        }
        lds_wave_sync();
    }
    if (sh.parts > 1u) __syncthreads();
    if (vok) {
#pragma unroll
        for (int s = 0; s < MS; ++s)
            if (s < n.S && (sh.parts == 1u || ((uint32_t)s & 3u) == sh.part) && L.del[s][lane] != 0)
                atomicAdd(&Y[ri.x_off + (uint64_t)s * N + v], (uint32_t)L.del[s][lane]);
    }
    opened_out = opened;
    return wave_ballot(big) != 0ull;
}

// Completes the leap of one tile (finish_counts) where the post-leap leap
// condition is judged: its violations too.  nx returns the lane's new counts
// (any sign).
template <int MS, int MR>
__device__ __forceinline__ void finish_tile(const KernelArgs& a, const NetView& n, const RealInfo& ri,
                                            cptr<RealCtl> cp, uint32_t t, uint32_t v0, uint32_t& bad, uint32_t& viol,
                                            uint32_t (&x)[MS], long long (&nx)[MS], bool judge) {
    const uint32_t v = v0 + (threadIdx.x & 63u);
#pragma unroll
    for (int s = 0; s < MS; ++s) {
        x[s] = 0u;
        nx[s] = 0;
    }
    if (v >= ri.N) return;
    uint32_t y[MS];
    bad = finish_counts<MS>(a, n.S, ri, wave_uniform(cp->cur), wave_uniform(cp->tgt), t, v, x, y, nx) ? 1u : 0u;
    if (judge) {
        const int c = n.C > 1 ? a.comp[ri.comp_off + v] : 0;
        double av[MR];
        uint32_t crit[(MR + 31) / 32];
        react_props<MR, MS>(n, x, c, a.n_critical, av, crit);
        viol = leap_condition_broken<MS, MR>(n, c, a.n_critical, a.epsilon, a.theta, x, nx, av, crit);
    }
}

// PartB::bad of two sets of tiles: bit 0 (a negative count) or-ed, the number
// of tiles beyond their queue above it added.
__device__ __forceinline__ uint32_t merge_bad(uint32_t p, uint32_t q) {
    return ((p & ~1u) + (q & ~1u)) | ((p | q) & 1u);
}

__device__ __forceinline__ void reduce_partB(unsigned long long& fire, uint32_t& bad, uint32_t& viol) {
    fire = wave_fold_u64(0ull, fire, [](unsigned long long p, unsigned long long q) { return p + q; });
    if (__ballot(bad != 0u) != 0ull) bad = wave_fold_u32(0u, bad, merge_bad);
    if (__ballot(viol != 0u) != 0ull)
        viol = wave_fold_u32(0u, viol, [](uint32_t p, uint32_t q) { return p + q; });
}

// Commits the step or leaps back, on c: returns true when the step was
// accepted and the realization runs on (its next step is then to be
// decided).  lead: the one thread that counts a finished realization in.
__device__ bool commit_step(const KernelArgs& a, const RealInfo& ri, unsigned long long fire, uint32_t bad,
                            uint32_t viol, RealCtl& c, bool lead) {
    if (bad >> 1 && lead) atomicAdd(a.redo_total, (unsigned long long)(bad >> 1));
    bad &= 1u;
    // A learned proposal is judged by Cao's leap condition after the fact: it
    // is kept only without negative populations and with no more violating
    // subvolumes than the plain method produces -- mean mu = viol_rate_max N,
    // with a Poisson upper bound mu + 3 sqrt(mu) + 2 so that small
    // realizations are not rejected for single violations; otherwise the
    // step is redone with Cao's tau and fresh draws.
    const double mu = a.viol_rate_max * (double)ri.N;
    const bool learned_reject = c.learned && (bad || (double)viol > mu + 3.0 * sqrt(mu) + 2.0);
    uint32_t z, w;
    spare_bufs(c.cur, c.tgt, z, w);
    if (bad || learned_reject) {
        c.attempt += 1u;
        if (learned_reject) {
            c.learned_rejects += 1;
            c.fallback = 1u;
            c.retry = 0u;
        } else {
            c.leapbacks += 1;
        }
        if (c.attempt > kMaxAttempt) {
            c.status = kErrLeapback;
            c.done = 1u;
            if (lead) atomicAdd(a.ndone, 1u);
            return false;
        }
        if (!learned_reject) {
            c.tau_p = c.tau_p * 0.5;
            decide(c);
            c.retry = 1u;
        }
        c.prop_ok = 0u;
        if (a.ep) c.tgt = w;
        return false;
    }
    // the leap pass of a learned context proposed the next step's tau from
    // the state it produced (edge-parallel pass only)
    c.prop_ok = a.props_in_finish ? 1u : 0u;
    const uint32_t old = c.cur;
    c.cur = c.tgt;
    c.tgt = a.ep ? z : old;
    c.t = c.last ? c.t_end : c.t + c.tau;
    c.step += 1u;
    c.steps += 1;
    c.firings += fire;
    c.subvolume_leaps += ri.N;
    c.violations += viol;
    if (c.crit) c.crit_events += 1;
    if (c.learned) c.learned_steps += 1;
    c.fallback = 0u;
    c.attempt = 0u;
    c.retry = 0u;
    if (c.t >= c.t_end || c.steps >= c.step_limit || c.t >= c.t_pause) {
        c.done = 1u;
        if (c.t >= c.t_end || c.steps >= c.step_limit) c.status = kDone;
        if (lead) atomicAdd(a.ndone, 1u);
        return false;
    }
    return true;
}

__device__ void finalize_B(const KernelArgs& a, const RealInfo& ri, uint32_t r, unsigned long long fire,
                           uint32_t bad, uint32_t viol, RealCtl c) {
    commit_step(a, ri, fire, bad, viol, c, true);
    a.ctl[r] = c;
}

__device__ __forceinline__ StepView step_view(const RealInfo& ri, cptr<RealCtl> cp) {
    StepView sv;
    sv.tau = cp->tau;
    sv.step = wave_uniform(cp->step);
    sv.attempt = wave_uniform(cp->attempt);
    sv.real = ri.id;
    sv.crit = (int)wave_uniform((uint32_t)cp->crit);
    sv.ev_kind = (int)wave_uniform((uint32_t)cp->ev_kind);
    sv.ev_idx = (int)wave_uniform((uint32_t)cp->ev_idx);
    sv.vstar = wave_uniform(cp->vstar);
    sv.ev_dst = wave_uniform(cp->ev_dst);
    return sv;
}

// The leap pass.  EP: the draws of every tile into the target buffer; the
// tile's firings go to its partial and the next pass completes the leap.  Otherwise one lane walks one subvolume's out- and in-edges and
// finishes it (networks beyond 8 species or 16 reactions, topologies beyond
// an entry's or a code's bits).  GEN: several compartments, or (EP) an
// asymmetric topology.
//
// The edge-parallel leap of 4 or 5 species, one compartment, runs at 5 waves
// per SIMD (96 VGPRs): at 6 the sampler spills (1M-subvolume Brusselator mesh
// 83.6 -> 94.5 us), at 4 fewer waves hide the walk's gathers (88 us).  Up to 3
// species draw dense tiles in the walk and run at 4 (at 5 it spills: bistable
// 64^3 grid 28.4 -> 29.6 us dense, 19.4 -> 20.9 sparse).
// SPLIT: a block of 4 wavefronts shares one tile, for contexts of few tiles,
// where one wavefront per tile leaves most SIMDs idle.
template <int MS, int MR, bool EP, bool GEN, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(EP && !GEN && MS <= 5 ? (MS <= 3 ? 4 : 5) : 1)))
void phase_b_kernel(KernelArgs a0) {
    const uint32_t wv = wave_uniform(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    __shared__ LeapLds<EP ? MS : 1, GEN> s_l[EP ? 4 : 1];  // (up to 4 waves per block)
    for (uint32_t it = 0;; ++it) {
        const uint32_t t = tile_at(it, a0.ntiles, SPLIT ? 1u : a0.waves_per_block, SPLIT ? 0u : wv);
        if (t == 0xFFFFFFFFu) break;
        const KernelArgs& a = tile_args();
        const NetView n = net_view<GEN>(a);
        const TileEnt te = ld_ro(a.tiles + t);
        const uint32_t r = wave_uniform(te.r);
        const RealInfo ri = ld_ro(a.info + r);
        const cptr<RealCtl> cp = ro(a.ctl + r);
        if (wave_uniform(cp->done)) continue;
        const StepView sv = step_view(ri, cp);
        const uint32_t* X = count_buf(a, wave_uniform(cp->cur));
        uint32_t* Xn = count_buf(a, wave_uniform(cp->tgt));
        unsigned long long fire = 0;
        uint32_t bad = 0, viol = 0;
        if constexpr (EP) {
            const TileShare<SPLIT ? 4u : 1u> sh{SPLIT ? wv : 0u};
            uint32_t opened = 0u;
            uint32_t big = leap_tile_draws<MS, MR, GEN>(a, n, ri, X, Xn, te.v0, sv, s_l[SPLIT ? 0u : wv], s_l[wv].q, sh,
                                                        fire, opened) ? 1u : 0u;
            reduce_partB(fire, bad, viol);
            if constexpr (SPLIT) {
                if (lane == 0) {
                    s_l[wv].part_fire = fire;
                    s_l[wv].part_opened = opened;
                    s_l[wv].part_big = big;
                }
                __syncthreads();
                for (uint32_t w = 1; wv == 0u && w < 4u; ++w) {
                    fire += s_l[w].part_fire;
                    opened += s_l[w].part_opened;
                    big |= s_l[w].part_big;
                }
            }
            if (lane == 0 && (!SPLIT || wv == 0u))
                a.partB_tile[t] = PartB{fire, (opened > kQueue || big) && a.count_redo ? 2u : 0u, 0u};
            if constexpr (SPLIT) __syncthreads();  // (before the next tile's staging)
        } else {
            const uint32_t v = te.v0 + lane;
            if (v < ri.N) bad = leap_subvolume<MS, MR>(a, n, ri, X, Xn, v, sv, fire, viol) ? 1u : 0u;
            reduce_partB(fire, bad, viol);
            if (lane == 0) a.partB_tile[t] = PartB{fire, bad, viol};
        }
    }
}

// The end of the edge-parallel leap pass of plain contexts that judge the
// post-leap leap condition (a check, off in ordinary runs): finish_tile in a
// pass of its own, so that the tau pass keeps its registers.
template <int MS, int MR, bool MC>
__global__ __launch_bounds__(256) void phase_b_finish_kernel(KernelArgs a) {
    const NetView n = net_view<MC>(a);
    const uint32_t lane = threadIdx.x & 63u;
    for (uint32_t it = 0;; ++it) {
        const uint32_t t = tile_at(it, a.ntiles, a.waves_per_block);
        if (t == 0xFFFFFFFFu) break;
        const TileEnt te = ld_ro(a.tiles + t);
        const uint32_t r = wave_uniform(te.r);
        const RealInfo ri = ld_ro(a.info + r);
        const cptr<RealCtl> cp = ro(a.ctl + r);
        if (wave_uniform(cp->done)) continue;
        unsigned long long fire = 0;
        uint32_t bad = 0, viol = 0;
        uint32_t x[MS];
        long long nx[MS];
        finish_tile<MS, MR>(a, n, ri, cp, t, te.v0, bad, viol, x, nx, true);
        reduce_partB(fire, bad, viol);
        if (lane == 0) {
            const PartB p = a.partB_tile[t];
            a.partB_tile[t] = PartB{p.fire, merge_bad(p.bad, bad), viol};
        }
    }
}

// Copies every running realization's counts to its target buffer, where the
// next edge-parallel leap adds its balances (the first kernel of a call: what
// was done to the buffers between calls does not matter).
static __global__ __launch_bounds__(256) void sync_target_kernel(KernelArgs a) {
    const uint32_t lane = threadIdx.x & 63u;
    for (uint32_t it = 0;; ++it) {
        const uint32_t t = tile_at(it, a.ntiles, a.waves_per_block);
        if (t == 0xFFFFFFFFu) break;
        const TileEnt te = ld_ro(a.tiles + t);
        const uint32_t r = wave_uniform(te.r);
        const RealInfo ri = ld_ro(a.info + r);
        const cptr<RealCtl> cp = ro(a.ctl + r);
        const uint32_t v = te.v0 + lane;
        if (wave_uniform(cp->done) || v >= ri.N) continue;
        const uint32_t* X = count_buf(a, wave_uniform(cp->cur)) + ri.x_off;
        uint32_t* Y = count_buf(a, wave_uniform(cp->tgt)) + ri.x_off;
        for (int s = 0; s < a.nh.S; ++s) Y[(uint64_t)s * ri.N + v] = X[(uint64_t)s * ri.N + v];
    }
}

// One block per realization: sum of firings / any negative over the tile
// partials of phase B, then commit the step or leap back.
static __global__ __launch_bounds__(1024) void commit_kernel(KernelArgs a) {
    const uint32_t r = blockIdx.x;
    if (r >= a.nreal) return;
    const RealInfo ri = ld_ro(a.info + r);
    const RealCtl c0 = ld_ro(a.ctl + r);
    if (c0.done) return;
    __shared__ unsigned long long s_f[16];
    __shared__ uint32_t s_b[16], s_v[16];
    unsigned long long fire = 0;
    uint32_t bad = 0, viol = 0;
    for (uint32_t q0 = 0; q0 < ri.ntiles; q0 += 8u * blockDim.x) {
        PartB p[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t q = q0 + (uint32_t)i * blockDim.x + threadIdx.x;
            p[i] = q < ri.ntiles ? a.partB_tile[ri.tile_begin + q] : PartB{0ull, 0u, 0u};
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            fire += p[i].fire;
            bad = merge_bad(bad, p[i].bad);
            viol += p[i].viol;
        }
    }
    reduce_partB(fire, bad, viol);
    const uint32_t wv = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    if (lane == 0) {
        s_f[wv] = fire;
        s_b[wv] = bad;
        s_v[wv] = viol;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (uint32_t w = 1; w < (blockDim.x >> 6); ++w) {
            fire += s_f[w];
            bad = merge_bad(bad, s_b[w]);
            viol += s_v[w];
        }
        finalize_B(a, ri, r, fire, bad, viol, c0);
    }
}

// The folded order of a plain-tau iteration: commits the step or leaps
// back from the leap pass's tile partials and, when the step is accepted
// and the realization runs on, decides the next step from the tile
// partials of the tau pass that ran on the new counts (phase_a_kernel with
// tau_spec) -- commit_kernel and decide_kernel in one launch.  Blocks and
// chunks as in decide_kernel (decide_chunks blocks per realization, the
// last one finishes; counter shared with decide_kernel, which never runs
// at the same time).  A leap-back drops the tau pass's partials (the
// retried leap reuses the halved tau).
template <int MS, int MR>
__global__ __launch_bounds__(decide_threads<MS>()) void commit_decide_kernel(KernelArgs a) {
    const uint32_t nch = a.decide_chunks;
    const uint32_t r = blockIdx.x / nch, chunk = blockIdx.x % nch;
    if (r >= a.nreal) return;
    const RealInfo ri = ld_ro(a.info + r);
    const RealCtl c0 = ld_ro(a.ctl + r);
    __shared__ unsigned long long s_f[16];
    __shared__ uint32_t s_b[16], s_v[16];
    __shared__ double s_tp[16], s_t2[16];
    __shared__ uint32_t s_v2[16];
    __shared__ uint32_t s_last;
    unsigned long long fire = 0ull;
    uint32_t bad = 0u, viol = 0u;
    double tp = kInf, t2 = kInf;
    uint32_t v2 = 0xFFFFFFFFu;
    const uint32_t per = (ri.ntiles + nch - 1u) / nch;
    const uint32_t qb = min(chunk * per, ri.ntiles), qe = min(qb + per, ri.ntiles);
    const PartB* pb = a.partB_tile + ri.tile_begin;
    const PartA* pa = a.partA_tile + ri.tile_begin;
    // both partials' loads in flight together
    for (uint32_t q0 = qb; q0 < qe; q0 += 8u * blockDim.x) {
        PartB b[8];
        PartA p[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t q = q0 + (uint32_t)i * blockDim.x + threadIdx.x;
            b[i] = q < qe ? pb[q] : PartB{0ull, 0u, 0u};
            p[i] = q < qe ? pa[q] : PartA{kInf, kInf, 0xFFFFFFFFu, 0u};
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            fire += b[i].fire;
            bad = merge_bad(bad, b[i].bad);
            viol += b[i].viol;
            merge_partA(tp, t2, v2, p[i].tp, p[i].t2, p[i].v2);
        }
    }
    if (c0.done) return;  // (the same in every block of the realization)
    reduce_partB(fire, bad, viol);
    const uint32_t wv = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    if (lane == 0) {
        s_f[wv] = fire;
        s_b[wv] = bad;
        s_v[wv] = viol;
    }
    reduce_block_partA<MS>(tp, t2, v2, s_tp, s_t2, s_v2);  // (its barrier publishes s_f / s_b / s_v)
    if (wv == 0)  // the first wavefront, every lane alike
        for (uint32_t w = 1; w < (blockDim.x >> 6); ++w) {
            fire += s_f[w];
            bad = merge_bad(bad, s_b[w]);
            viol += s_v[w];
        }
    if (nch > 1u) {
        if (threadIdx.x == 0) {
            a.partA_chunk[r * nch + chunk] = PartA{tp, t2, v2, 0u};
            a.partB_chunk[r * nch + chunk] = PartB{fire, bad, viol};
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            s_last = atomicAdd(&a.decide_cnt[r], 1u) == nch - 1u ? 1u : 0u;
        }
        __syncthreads();
        if (!s_last || wv != 0) return;
        // the last block of the realization: its first wavefront finishes
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        PartA p{kInf, kInf, 0xFFFFFFFFu, 0u};
        PartB b{0ull, 0u, 0u};
        if (lane < nch) {
            p = a.partA_chunk[r * nch + lane];
            b = a.partB_chunk[r * nch + lane];
        }
        tp = p.tp;
        t2 = p.t2;
        v2 = p.v2;
        fire = b.fire;
        bad = b.bad;
        viol = b.viol;
        reduce_partA(tp, t2, v2);
        reduce_partB(fire, bad, viol);
        if (lane == 0) a.decide_cnt[r] = 0u;
    } else if (wv != 0) {
        return;
    }
    RealCtl c = c0;
    if (!commit_step(a, ri, fire, bad, viol, c, lane == 0u)) {
        if (lane == 0u) a.ctl[r] = c;
        return;
    }
    finalize_A<MS, MR>(a, net_view(a), ri, r, tp, t2, v2, c);
}

}  // namespace plis
