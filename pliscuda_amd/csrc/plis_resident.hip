// plis_resident.hip -- all steps of a small realization inside one block.
//
// Stepping a small realization with one launch per pass is bound by launches:
// a kernel of the captured step that finds nothing to do takes 4.4 us with what
// its boundary flushes (1.65 in a graph of empty kernels), the whole step of a
// 64-subvolume box 26-29 us whatever its size.  resident_kernel gives each
// realization one block that makes up to `iters` iterations: counts,
// balances and propensities stay in LDS (in a global workspace for networks
// of many species that do not fit), passes are separated by block barriers,
// and the step is decided and committed by the first wavefront.  What bounds
// it is the latency of six dependent phases per step on one CU.
//
// A phase hands out wavefront-sized items -- (reaction, tile), (species,
// tile), (hop block, 64 forward entries) -- so that a box of one tile still
// fills several wavefronts and every table index stays wave-uniform; the
// launch-per-pass kernels, one lane per subvolume with all species in
// registers, leave a 60-subvolume realization of 32 species one wavefront
// that walks everything serially out of scratch memory.
//
// Every value is formed by the same operations in the same order as in the
// launch-per-pass kernels (propensities, the FP64 sums of tau', draw words),
// so a trajectory does not depend on which of them runs.
#include "plis_kernels.hip"
#include "plis_resident.h"

namespace plis {

constexpr uint32_t kResReact = 0x80000000u;  // reaction code: flag | subvolume << 7 | j; hop: entry << 7 | w

// The items (hi, lo), lo < m, of a phase that fall to wavefront wv of nw:
// hi is the table index, lo the tile or the group of 64 entries.
struct ResItems {
    uint32_t hi, lo, dh, dl, m;
    __device__ __forceinline__ ResItems(uint32_t wv, uint32_t nw, uint32_t m_) : m(m_) {
        hi = wv / m;
        lo = wv % m;
        dh = nw / m;
        dl = nw % m;
    }
    __device__ __forceinline__ void next() {
        hi += dh;
        lo += dl;
        if (lo >= m) {
            lo -= m;
            ++hi;
        }
    }
};

// Network tables in LDS, copied once per launch: a table entry then costs an
// LDS read where the scalar cache costs several times as much.
struct ResTables {
    const double *k, *d;   // [c R + j], [c S + s]
    const int4* rx;        // reaction j: {reactants | (order > 0) << 8, species x 3}, {multiplicities x 3, 0}
    const int2 *sp, *spe;  // species s: {first, end} of its entries {reaction, change}
    const int2 *jp, *jpe;  // reaction j: {first, end} of its entries {species, change}
    const int2* hm;        // species s: {highest order, multiplicity}
};

// A block's view of its realization.  prop: propensities [j N + v], the sign
// bit set where the reaction is critical; del: balances of the step; x, xn:
// counts and the counts the step makes; fwd: forward entries {upper end,
// weight, lower end, weight back}; in / inp: in-edges {id, weight} and their
// row pointers.
struct ResView {
    double* prop;
    unsigned long long* del;
    uint32_t *x, *xn;
    const uint4* fwd;
    const uint2* in;
    const uint32_t* inp;
    const double* wsum;
    const int32_t* comp;  // (several compartments only)
    ResTables t;
    uint32_t N, S, R;
    bool mc;
};

struct ResStep {
    double tau;
    float tauf;
    uint32_t step, c3react, c3hop;
};

// A draw its coarse byte leaves open, complete sampler, applied to the
// balances; returns the firings.
__device__ __forceinline__ long long res_draw(const KernelArgs& a, const ResView& R, const ResStep& st, uint32_t code,
                                              uint32_t hb) {
    const bool react = (code & kResReact) != 0u;
    const uint32_t w = code & 127u, s = w >> 1;
    uint32_t c0, c1, c3;
    double lam;
    float lf;
    if (react) {
        c0 = (code >> 7) & 0xFFFFFFu;
        c1 = kSelfId;
        c3 = st.c3react;
        lam = st.tau * __builtin_fabs(R.prop[w * R.N + c0]);
        lf = (float)lam;
    } else {
        const uint4 f = R.fwd[(code >> 7) & 0xFFFFFFu];
        c0 = f.z;
        c1 = f.x;
        c3 = st.c3hop;
        const bool back = (w & 1u) != 0u;
        const uint32_t from = back ? c1 : c0;
        const float wf = __uint_as_float(back ? f.w : f.y);
        const double d = R.t.d[(R.mc ? (uint32_t)R.comp[from] : 0u) * R.S + s];
        const uint32_t xs = R.x[s * R.N + from];
        lam = hop_mean(d, xs, (double)wf, st.tau, a.n_critical);
        lf = hop_mean_f(d, xs, wf, st.tauf, a.n_critical);
    }
    const uint32_t fb = c3 | (kFineBlock + (w >> 2));
    const uint32_t word = draw_word(hb, philox10(c0, c1, st.step, fb, a.seed_lo, a.seed_hi), w);
    long long k = lf < kSqueezeMaxF ? poisson_squeeze(lf, __uint2float_rn(word) * 0x1p-32f) : -1;
    if (k < 0) k = poisson_slow(lam, word, DrawId{c0, c1, st.step, fb, a.seed_lo, a.seed_hi, w & 3u});
    if (k == 0) return 0;
    if (react) {
        const int2 p = R.t.jp[w];
        for (int e = p.x; e < p.y; ++e) {
            const int2 ch = R.t.jpe[e];
            atomicAdd(&R.del[(uint32_t)ch.x * R.N + c0], (unsigned long long)(k * (long long)ch.y));
        }
    } else {
        const long long b = (w & 1u) ? k : -k;  // balance of the entry's lower end
        atomicAdd(&R.del[s * R.N + c0], (unsigned long long)b);
        atomicAdd(&R.del[s * R.N + c1], (unsigned long long)-b);
    }
    return k;
}

// The critical event at c.vstar on counts x, as choose_event picks it.
__device__ void res_choose_event(const KernelArgs& a, const NetView& n, const RealInfo& ri, RealCtl& c,
                                 const double* prop, const uint32_t* x) {
    const uint32_t v = c.vstar, N = ri.N;
    const HopRow row = hop_row(a, ri, v);
    const int cc = n.C > 1 ? a.comp[ri.comp_off + v] : 0;
    const double W = a.wsum[ri.rp_off + v];
    double a0c = 0.0;
    for (int j = 0; j < n.R; ++j) {
        const double p = prop[(uint32_t)j * N + v];
        if (__builtin_signbit(p)) a0c += -p;
    }
    for (int s = 0; s < n.S; ++s) {
        const double d = n.d[cc * n.S + s];
        const uint32_t xs = x[(uint32_t)s * N + v];
        if (d > 0.0 && !hop_active(d, xs, a.n_critical)) a0c += (d * (double)xs) * W;
    }
    const U4 o = philox10(v, kSelfId, c.step, ctr_word3(ri.id, 0u, kCrit, 0u), a.seed_lo, a.seed_hi);
    const double target = uniform01(o.x) * a0c;
    double acc = 0.0;
    int kind = 0, idx = -1;
    for (int j = 0; j < n.R; ++j) {
        const double p = prop[(uint32_t)j * N + v];
        if (!__builtin_signbit(p) || !(-p > 0.0)) continue;
        acc += -p;
        idx = j;
        if (target < acc) {
            kind = 1;
            break;
        }
    }
    int lastkind = idx >= 0 ? 1 : 0;
    if (kind == 0) {
        for (int s = 0; s < n.S; ++s) {
            const double d = n.d[cc * n.S + s];
            const uint32_t xs = x[(uint32_t)s * N + v];
            if (!(d > 0.0) || hop_active(d, xs, a.n_critical)) continue;
            const double ao = (d * (double)xs) * W;
            if (!(ao > 0.0)) continue;
            acc += ao;
            idx = s;
            lastkind = 2;
            if (target < acc) {
                kind = 2;
                break;
            }
        }
    }
    if (kind == 0) kind = lastkind;
    c.ev_kind = kind;
    c.ev_idx = idx;
    c.ev_dst = kind == 2 ? choose_hop_edge(a, ri, v, row.rb, row.re, row.cw, uniform01(o.y) * W) : v;
}

// MODE 0: everything in LDS; 1: the topology stays in global memory; 2: the
// arrays too (a workspace).
template <int MODE>
static __global__ __launch_bounds__(1024) void resident_kernel(ResidentArgs ra) {
    extern __shared__ __align__(16) unsigned char s_dyn[];
    __shared__ RealCtl s_c;
    __shared__ double s_tp[16], s_t2[16];
    __shared__ uint32_t s_v2[16];
    __shared__ unsigned long long s_fire;
    __shared__ uint32_t s_bad;
    const KernelArgs& a = ra.k;
    const uint32_t r = blockIdx.x;
    const RealInfo ri = ld_ro(a.info + r);
    const RealCtl c0 = ld_ro(a.ctl + r);
    if (c0.done) return;
    const uint32_t lane = threadIdx.x & 63u, wv = wave_uniform(threadIdx.x >> 6), nw = blockDim.x >> 6;
    const uint32_t N = ri.N, nt = ri.ntiles;
    const NetView n = net_view(a);
    const uint32_t S = (uint32_t)n.S, R = (uint32_t)n.R, C = (uint32_t)n.C;
    const int nc = a.n_critical;
    const uint32_t nc1 = nc > 1 ? (uint32_t)nc : 1u;
    const uint32_t nf = a.frp[ri.rp_off + N];  // forward entries
    const bool sym = (ri.flags & 1u) != 0;
    const uint64_t* const g_in = sym ? a.cw + ri.e_off : a.icw + ri.ie_off;
    const uint32_t* const g_inp = sym ? a.rp + ri.rp_off : a.irp + ri.irp_off;

    // LDS: queues, tile counters, tables, then (MODE 0, 1) the arrays and
    // (MODE 0) the topology; resident_lds() adds up the same
    uint32_t at = 0u;
    auto take = [&](uint32_t bytes) {
        const uint32_t o = at;
        at += (bytes + 15u) & ~15u;
        return s_dyn + o;
    };
    uint2* const q = reinterpret_cast<uint2*>(take(nw * kResidentQueue * 8u)) + wv * kResidentQueue;
    uint32_t* const tcnt = reinterpret_cast<uint32_t*>(take(nt * 4u));
    ResView V;
    V.N = N;
    V.S = S;
    V.R = R;
    V.mc = C > 1u;
    {
        auto copy = [&](auto* from, uint32_t count) {
            using T = std::remove_cv_t<std::remove_pointer_t<decltype(from)>>;
            T* to = reinterpret_cast<T*>(take(count * (uint32_t)sizeof(T)));
            for (uint32_t i = threadIdx.x; i < count; i += blockDim.x) to[i] = from[i];
            return (const T*)to;
        };
        V.t.k = copy(a.net_d + a.nh.off_k, C * R);
        V.t.d = copy(a.net_d + a.nh.off_d, C * S);
        V.t.rx = copy(ra.rx, 2u * R);
        V.t.sp = copy(ra.sp, S);
        V.t.spe = copy(ra.spe, ra.nspe);
        V.t.jp = copy(ra.jp, R);
        V.t.jpe = copy(ra.jpe, ra.nspe);
        V.t.hm = copy(ra.hm, S);
        unsigned char* base;
        if constexpr (MODE == 2) base = reinterpret_cast<unsigned char*>(ra.ws) + (uint64_t)r * ra.ws_slice;
        else base = take(N * (8u * R + 16u * S));
        V.prop = reinterpret_cast<double*>(base);
        V.del = reinterpret_cast<unsigned long long*>(V.prop + R * N);
        V.x = reinterpret_cast<uint32_t*>(V.del + S * N);
        V.xn = V.x + S * N;
        if constexpr (MODE == 0) {
            V.wsum = copy(a.wsum + ri.rp_off, N);
            V.fwd = copy(ra.fwd + ri.fe_off, nf);
            V.inp = copy(g_inp, N + 1u);
            V.in = copy(reinterpret_cast<const uint2*>(g_in), g_inp[N]);
            V.comp = V.mc ? copy(a.comp + ri.comp_off, N) : nullptr;
        } else {
            V.wsum = a.wsum + ri.rp_off;
            V.fwd = ra.fwd + ri.fe_off;
            V.inp = g_inp;
            V.in = reinterpret_cast<const uint2*>(g_in);
            V.comp = a.comp + ri.comp_off;
        }
        const uint32_t* X = count_buf(a, c0.cur);
        for (uint32_t i = threadIdx.x; i < S * N; i += blockDim.x) {
            V.x[i] = X[ri.x_off + i];
            V.del[i] = 0ull;
        }
        for (uint32_t t = threadIdx.x; t < nt; t += blockDim.x) tcnt[t] = 0u;
        if (threadIdx.x == 0u) {
            s_c = c0;
            s_fire = 0ull;
            s_bad = 0u;
        }
    }
    uint32_t* const xb = V.x;
    uint32_t cb = 0u;  // count buffer in use: xb + cb S N
    uint32_t cur = c0.cur;

    auto props = [&](const uint32_t* x) {
        for (ResItems it(wv, nw, nt); it.hi < R; it.next()) {
            const uint32_t j = it.hi, v = it.lo * 64u + lane, vq = min(v, N - 1u);
            const int4 r0 = V.t.rx[2u * j], r1 = V.t.rx[2u * j + 1u];
            const uint32_t nr = wave_uniform((uint32_t)r0.x);
            const uint32_t x0 = x[(uint32_t)r0.y * N + vq], x1 = x[(uint32_t)r0.z * N + vq], x2 = x[(uint32_t)r0.w * N + vq];
            double aj = V.t.k[(V.mc ? (uint32_t)V.comp[vq] : 0u) * R + j];
            bool low = false;
            auto reactant = [&](uint32_t xs, int m) {
                m = (int)wave_uniform((uint32_t)m);
                aj = aj * binom_d(xs, m);
                low = low || below_nc(xs, m, nc);
            };
            if ((nr & 255u) > 0u) reactant(x0, r1.x);
            if ((nr & 255u) > 1u) reactant(x1, r1.y);
            if ((nr & 255u) > 2u) reactant(x2, r1.z);
            if (v < N) V.prop[j * N + v] = (nr & 256u) && low ? -aj : aj;
        }
    };
    // tau' per (species, tile) and tau'' per tile into the wavefront's slot
    auto taus = [&](const uint32_t* x, uint32_t step) {
        double tp = kInf, t2 = kInf;
        uint32_t v2 = 0xFFFFFFFFu;
        for (ResItems it(wv, nw, nt); it.hi <= S; it.next()) {
            const uint32_t v = it.lo * 64u + lane;
            if (it.hi == S) {
                if (v >= N) continue;
                double a0c = 0.0;
#pragma unroll 4
                for (uint32_t j = 0; j < R; ++j) {
                    const double p = V.prop[j * N + v];
                    a0c += __builtin_signbit(p) ? -p : 0.0;
                }
                const uint32_t c = V.mc ? (uint32_t)V.comp[v] : 0u;
                const double W = V.wsum[v];
                for (uint64_t m = ra.diffusing; m != 0u; m &= m - 1u) {
                    const uint32_t s = (uint32_t)__builtin_ctzll(m);
                    const double d = V.t.d[c * S + s];
                    const uint32_t xs = x[s * N + v];
                    if (d > 0.0 && !hop_active(d, xs, nc)) a0c += (d * (double)xs) * W;
                }
                if (a0c > 0.0) {
                    const U4 o = philox10(v, kSelfId, step, ctr_word3(ri.id, 0u, kTau2, 0u), a.seed_lo, a.seed_hi);
                    const double t = -dlog(uniform01(o.x)) / a0c;
                    if (t < t2 || (t == t2 && v < v2)) {
                        t2 = t;
                        v2 = v;
                    }
                }
                continue;
            }
            const uint32_t s = it.hi;
            const int2 hm = V.t.hm[s];
            const int hor = (int)wave_uniform((uint32_t)hm.x);
            if (hor == 0 || v >= N) continue;
            double mu = 0.0, sig = 0.0;
            const int2 sp = V.t.sp[s];
            const int e1 = (int)wave_uniform((uint32_t)sp.y);
#pragma unroll 4
            for (int e = (int)wave_uniform((uint32_t)sp.x); e < e1; ++e) {
                const int2 ch = V.t.spe[e];
                const double p = V.prop[(uint32_t)ch.x * N + v];
                const double pa = __builtin_signbit(p) ? 0.0 : p;  // a critical reaction adds 0
                mu += (double)ch.y * pa;
                sig += (double)(ch.y * ch.y) * pa;
            }
            const uint32_t xs = x[s * N + v];
            if ((ra.diffusing >> s) & 1u) {
                const double d = V.t.d[(V.mc ? (uint32_t)V.comp[v] : 0u) * S + s];
                if (hop_active(d, xs, nc)) {
                    const double aout = (d * (double)xs) * V.wsum[v];
                    mu -= aout;
                    sig += aout;
                }
                // four in-edges at once (their loads in flight together); one
                // past the row's end adds +0
                const uint32_t ie = V.inp[v + 1u];
                for (uint32_t e = V.inp[v]; e < ie; e += 4u) {
                    double ain[4];
                    uint2 cw[4];
#pragma unroll
                    for (uint32_t i = 0; i < 4u; ++i) cw[i] = V.in[min(e + i, ie - 1u)];
#pragma unroll
                    for (uint32_t i = 0; i < 4u; ++i) {
                        const uint32_t xu = x[s * N + cw[i].x];
                        const double du = V.mc ? V.t.d[(uint32_t)V.comp[cw[i].x] * S + s] : d;
                        ain[i] = (du * (double)(xu >= nc1 && e + i < ie ? xu : 0u)) * (double)__uint_as_float(cw[i].y);
                    }
#pragma unroll
                    for (uint32_t i = 0; i < 4u; ++i) {
                        mu += ain[i];
                        sig += ain[i];
                    }
                }
            }
            const double mm = fmax(eps_x_over_g(a.epsilon, hor, (int)wave_uniform((uint32_t)hm.y), xs), 1.0);
            tp = fmin(tp, fmin(mm / __builtin_fabs(mu), (mm * mm) / sig));
        }
        reduce_partA(tp, t2, v2);
        if (lane == 0u) {
            s_tp[wv] = tp;
            s_t2[wv] = t2;
            s_v2[wv] = v2;
        }
    };
    // the step decision from the wavefronts' slots (first wavefront)
    auto finalize = [&](RealCtl& c, const uint32_t* x) {
        double tp = lane < nw ? s_tp[lane] : kInf, t2 = lane < nw ? s_t2[lane] : kInf;
        uint32_t v2 = lane < nw ? s_v2[lane] : 0xFFFFFFFFu;
        reduce_partA(tp, t2, v2);
        if (tp == kInf && t2 == kInf) {
            c.status = kAbsorbed;
            c.done = 1u;
            if (lane == 0u) atomicAdd(a.ndone, 1u);
            return;
        }
        c.tau_p = tp;
        c.tau2 = t2;
        c.vstar = v2;
        c.learned = 0u;
        c.ev_kind = 0;
        c.ev_idx = -1;
        c.ev_dst = v2;
        decide(c);
        if (t2 < kInf && t2 <= tp) res_choose_event(a, n, ri, c, V.prop, x);
    };

    __syncthreads();
    props(xb);
    __syncthreads();
    if (!c0.retry) {  // a retried leap keeps its halved tau
        taus(xb, c0.step);
        __syncthreads();
        if (wv == 0u) {
            RealCtl c = c0;
            finalize(c, xb);
            if (lane == 0u) s_c = c;
        }
        __syncthreads();
    }

    for (uint32_t iter = 0; iter < ra.iters && !s_c.done; ++iter) {
        V.x = xb + cb * S * N;
        V.xn = xb + (cb ^ 1u) * S * N;
        // draws: an item is 8 species' hops of 64 forward entries or 4
        // reactions of a tile.  The lanes' open draws enter the wavefront's
        // queue one per lane and round; it is drawn when the next round might
        // not fit, and at the end.
        {
            ResStep st;
            st.tau = s_c.tau;
            st.tauf = (float)st.tau;
            st.step = wave_uniform(s_c.step);
            const uint32_t attempt = wave_uniform(s_c.attempt);
            st.c3react = ctr_word3(ri.id, attempt, kReact, 0u);
            st.c3hop = ctr_word3(ri.id, attempt, kHop, 0u);
            unsigned long long fire = 0ull;
            uint32_t qn = 0u;
            const uint32_t nch = (nf + 63u) >> 6, hops = nch * ((S + 7u) >> 3), items = hops + nt * ((R + 3u) >> 2);
            uint32_t item = wv;
            uint32_t open = 0u, code = 0u;  // open draws of the item: bit b is draw code + b
            U4 o{0u, 0u, 0u, 0u};
            for (;;) {
                while (__ballot(open != 0u) == 0ull && item < items) {
                    uint32_t cnt = 0u, tile = 0u;
                    if (item < hops) {
                        const uint32_t b = item / nch, e = (item % nch) * 64u + lane;
                        uint32_t m = (uint32_t)(ra.diffusing >> (8u * b)) & 0xFFu;
                        if (m != 0u) {
                            const uint4 f = V.fwd[min(e, nf - 1u)];
                            const uint32_t v = f.z, u = f.x;
                            const uint32_t dv = V.mc ? (uint32_t)V.comp[v] * S : 0u, du = V.mc ? (uint32_t)V.comp[u] * S : 0u;
                            o = philox10(v, u, st.step, st.c3hop | b, a.seed_lo, a.seed_hi);
                            for (; m != 0u; m &= m - 1u) {
                                const uint32_t sl = (uint32_t)__builtin_ctz(m), s = 8u * b + sl;
                                const uint32_t xo = V.x[s * N + v], xu = V.x[s * N + u];
                                const double d0 = V.t.d[dv + s], d1 = V.t.d[du + s];
#pragma unroll
                                for (uint32_t dir = 0; dir < 2u; ++dir) {
                                    const float lf = hop_mean_f(dir ? d1 : d0, dir ? xu : xo,
                                                                __uint_as_float(dir ? f.w : f.y), st.tauf, nc);
                                    const float hb = (float)coarse_byte(o, 2u * sl + dir);
                                    if (hb > coarse_bound(lf)) {
                                        open |= 1u << (2u * sl + dir);
                                        cnt += lf > kPtrsMaybeF ? kQueue + 1u : 1u;
                                    }
                                }
                            }
                            if (e >= nf) open = cnt = 0u;
                            code = (e << 7) | (16u * b);
                            tile = v >> 6;
                        }
                    } else {
                        const uint32_t g = (item - hops) / nt, j0 = 4u * g;
                        tile = (item - hops) % nt;
                        const uint32_t v = tile * 64u + lane, vq = min(v, N - 1u);
                        o = philox10(v, kSelfId, st.step, st.c3react | (j0 >> 4), a.seed_lo, a.seed_hi);
#pragma unroll
                        for (uint32_t b = 0; b < 4u; ++b) {
                            if (j0 + b >= R) break;
                            const double p = V.prop[(j0 + b) * N + vq];
                            const double lam = st.tau * p;
                            if (!__builtin_signbit(p) && p > 0.0 && !coarse_zero(lam, coarse_byte(o, j0 + b))) {
                                open |= 1u << b;
                                cnt += lam < kPoissonInvMax ? 1u : kQueue + 1u;
                            }
                        }
                        if (v >= N) open = cnt = 0u;
                        code = kResReact | (v << 7) | j0;
                    }
                    if (a.count_redo && cnt != 0u) atomicAdd(&tcnt[tile], cnt);
                    item += nw;
                }
                const unsigned long long any = __ballot(open != 0u);
                const uint32_t cnt = (uint32_t)__popcll(any);
                if (cnt == 0u || qn + cnt > kResidentQueue) {
                    lds_wave_sync();
                    for (uint32_t i = lane; i < qn; i += 64u)
                        fire += (unsigned long long)res_draw(a, V, st, q[i].x, q[i].y);
                    lds_wave_sync();
                    qn = 0u;
                    if (cnt == 0u) break;
                }
                if (open != 0u) {
                    const uint32_t c = code + (uint32_t)__builtin_ctz(open);
                    open &= open - 1u;
                    q[qn + __builtin_amdgcn_mbcnt_hi((uint32_t)(any >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)any, 0u))] =
                        make_uint2(c, coarse_byte(o, c & 15u));
                }
                qn += cnt;
            }
            if (fire != 0ull) atomicAdd(&s_fire, fire);
        }
        __syncthreads();
        // new counts
        {
            const int kind = s_c.crit ? s_c.ev_kind : 0;
            const int idx = s_c.ev_idx;
            const uint32_t vstar = s_c.vstar, dst = s_c.ev_dst;
            bool bad = false;
            for (ResItems it(wv, nw, nt); it.hi < S; it.next()) {
                const uint32_t v = it.lo * 64u + lane;
                if (v >= N) continue;
                const uint32_t i = it.hi * N + v;
                long long y = (long long)V.x[i] + (long long)V.del[i];
                V.del[i] = 0ull;
                if (kind == 1 && v == vstar) y += n.nu[it.hi * R + (uint32_t)idx];
                if (kind == 2 && (int)it.hi == idx) {
                    if (v == vstar) y -= 1;
                    if (v == dst && dst != vstar) y += 1;
                }
                bad = bad || y < 0 || y > 0xFFFFFFFFll;
                V.xn[i] = (uint32_t)y;
            }
            if (bad) s_bad = 1u;
            if (a.count_redo)
                for (uint32_t t = threadIdx.x; t < nt; t += blockDim.x) {
                    if (tcnt[t] > kQueue) atomicAdd(a.redo_total, 1ull);
                    tcnt[t] = 0u;
                }
        }
        __syncthreads();
        props(V.xn);
        __syncthreads();
        taus(V.xn, s_c.step + 1u);
        __syncthreads();
        if (wv == 0u) {
            RealCtl c = s_c;
            unsigned long long fire = s_fire;
            if (c.crit && (c.ev_kind == 1 || c.ev_kind == 2)) fire += 1ull;
            if (commit_step(a, ri, fire, s_bad, 0u, c, lane == 0u)) finalize(c, V.xn);
            lds_wave_sync();
            if (lane == 0u) {
                s_c = c;
                s_fire = 0ull;
                s_bad = 0u;
            }
        }
        __syncthreads();
        if (s_c.cur != cur) {
            cur = s_c.cur;
            cb ^= 1u;
        } else {  // leap-back: the propensities of the counts before the step again
            props(V.x);
            __syncthreads();
        }
    }
    uint32_t* X = count_buf(a, s_c.cur);
    for (uint32_t i = threadIdx.x; i < S * N; i += blockDim.x) X[ri.x_off + i] = xb[cb * S * N + i];
    if (threadIdx.x == 0u) a.ctl[r] = s_c;
}

hipError_t resident_reserve(uint32_t lds) {
    hipError_t e = hipSuccess;
    for (const void* k : {reinterpret_cast<const void*>(&resident_kernel<0>), reinterpret_cast<const void*>(&resident_kernel<1>),
                          reinterpret_cast<const void*>(&resident_kernel<2>)})
        if (e == hipSuccess) e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    return e;
}

hipError_t launch_resident(hipStream_t stream, uint32_t nreal, uint32_t waves, uint32_t lds, int mode,
                           const ResidentArgs& ra) {
    const dim3 grid(nreal), block(64u * waves);
    switch (mode) {
        case 0: hipLaunchKernelGGL(resident_kernel<0>, grid, block, lds, stream, ra); break;
        case 1: hipLaunchKernelGGL(resident_kernel<1>, grid, block, lds, stream, ra); break;
        default: hipLaunchKernelGGL(resident_kernel<2>, grid, block, lds, stream, ra); break;
    }
    return hipGetLastError();
}

}  // namespace plis
