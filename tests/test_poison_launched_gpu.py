"""The initcheck stand-in where every pass is a launch: contexts too large for the
one-block kernel, or stepped with plis_profile, which launches every pass.  Every
buffer that a step writes before it reads is poisoned before each call; calls of
single iterations end after accepted steps and after leap-backs.  A poisoned run
must equal a clean one and the oracle bit for bit."""
import numpy as np
import pytest

from oracle import ffi
from pliscuda_amd import capi
from pliscuda_amd import workloads as W
from tests import helpers as H

pytestmark = pytest.mark.gpu

FIELDS = ("steps", "leapbacks", "firings", "crit_events", "t")


def _chain(S):
    sp = [f"X{i}" for i in range(S)]
    return W.network(sp, [({sp[i]: 1}, {sp[(i + 1) % S]: 1}) for i in range(S)] + [({sp[0]: 1, sp[1]: 1}, {sp[2]: 1}), ({}, {sp[0]: 2})],
                     [0.4] * S + [2e-3, 3.0], [0.5 if i % 3 == 0 else 0.0 for i in range(S)])


def _large(name):
    """(network, topologies, counts, epsilon, n_c): beyond the one-block kernel's sizes"""
    abc = W.abc_network()
    if name == "mesh":  # five species, a launch per pass from about 450 subvolumes
        t = W.random_mesh(12, 10, 10, 4)
        return W.brusselator_network(W.SEED_BRUSS), [t], [W.poisson_state(5, t["N"], [60, 40, 80, 100, 20], 5)], 0.03, 10
    if name == "asym":
        t = H.asym_topology(2001, 3)
        return abc, [t], [W.poisson_state(3, t["N"], 30.0, 5)], 0.03, 10
    if name == "compartments":
        t = dict(W.cubic_grid(13, 13, 11, periodic=False))
        t["comp"] = (np.arange(t["N"]) % 3 == 0).astype(np.int32)
        return H.two_compartment_case()[0], [t], [W.poisson_state(3, t["N"], 30.0, 5)], 0.03, 10
    if name == "wide":  # balances of thousands of molecules
        t = W.cubic_grid(13, 13, 11, periodic=False)
        net = W.network(["A"], [({"A": 1}, {"A": 1})], [0.0], [5.0])
        return net, [t], [W.uniform_state(t["N"], 299_000, 301_000, 3)], 0.05, 10
    if name in ("leapback", "leapback_asym"):
        t = H.asym_topology(2000, 3) if name.endswith("asym") else W.cubic_grid(13, 13, 11, periodic=False)
        return abc, [t], [W.poisson_state(3, t["N"], [2.0, 2.0, 1.0], 8)], 0.9, 0
    if name == "critical":
        t = W.cubic_grid(13, 13, 11, periodic=False)
        return abc, [t], [W.poisson_state(3, t["N"], [11.0, 11.0, 9.0], 8)], 0.03, 10
    if name == "uneven":
        ts = [W.cubic_grid(*s, periodic=False) for s in ((12, 12, 9), (3, 3, 2), (7, 8, 5))]
        return abc, ts, [W.poisson_state(3, t["N"], 30.0, i) for i, t in enumerate(ts)], 0.03, 10
    if name == "general":  # 20 species: the per-subvolume leap
        t = W.cubic_grid(20, 20, 20, periodic=False)
        return _chain(20), [t], [W.poisson_state(20, t["N"], 30.0, 7)], 0.03, 10
    if name == "split_off":  # more than 1,024 tiles: a wavefront per tile of the leap
        t = W.cubic_grid(41, 41, 40, periodic=False)
        return abc, [t], [W.poisson_state(3, t["N"], [40.0, 12.0, 30.0], 8)], 0.1, 10
    raise KeyError(name)


def _small(name):
    """One-block sizes, stepped with plis_profile."""
    abc = W.abc_network()
    if name == "mesh":
        net, t, x = H.small_bruss()
        return net, [t], [x], 0.03, 10
    if name == "asym":
        net, t, _ = H.small_bruss()
        t = H.asym_topology(t["N"], 3)
        return net, [t], [W.poisson_state(5, t["N"], 60.0, 3)], 0.03, 10
    if name == "critical":
        net, t, x = H.low_count_case()
        return net, [t], [x], 0.03, 10
    if name == "leapback":
        net, t, x = H.low_count_case(seed=23)
        return net, [t], [x], 0.9, 2
    if name == "uneven":
        ts = [W.cubic_grid(*s, periodic=False) for s in ((5, 4, 3), (1, 1, 1), (8, 8, 2))]
        return abc, ts, [W.poisson_state(3, t["N"], 30.0, i) for i, t in enumerate(ts)], 0.03, 10
    if name == "general":
        t = W.cubic_grid(19, 2, 2, periodic=False)
        return _chain(20), [t], [W.poisson_state(20, t["N"], 30.0, 7)], 0.03, 10
    raise KeyError(name)


def _compare(case, calls, step, seed=9):
    net, topos, xs, eps, nc = case
    out = []
    for poison in (False, True):
        ctx = capi.Context(net, topos, xs, eps=eps, nc=nc, seed=seed)
        ctx.arm()
        after_back, backs = 0, 0
        for n in calls:
            if poison:
                ctx.debug_poison()
            step(ctx, n)
            b = sum(ctx.stats(r)["leapbacks"] for r in range(ctx.n))
            after_back += n == 1 and b > backs
            backs = b
        out.append(([ctx.get_state(r) for r in range(ctx.n)], [ctx.stats(r) for r in range(ctx.n)]))
        ctx.close()
    (xa, sa), (xb, sb) = out
    for r, t in enumerate(topos):
        assert np.array_equal(xa[r], xb[r]), f"realization {r}: state differs after poisoning"
        assert all(sa[r][f] == sb[r][f] for f in FIELDS)
        x = np.array(xs[r], dtype=np.uint32).copy()
        so = ffi.run(ffi.Model(net, t), x, eps, nc, seed, np.inf, step_limit=sa[r]["steps"], realization=r)
        # (a leap-back after the last accepted step is the GPU's alone)
        assert np.array_equal(xa[r], x) and sa[r]["t"] == so.t and sa[r]["firings"] == so.firings
        assert sa[r]["steps"] + sa[r]["leapbacks"] == sum(calls)
    return sa, after_back


@pytest.mark.parametrize("name", ["mesh", "asym", "compartments", "wide", "critical", "uneven", "general", "split_off"])
def test_large_contexts(name):
    sa, _ = _compare(_large(name), (1, 4, 2, 5), lambda ctx, n: ctx.iterate(n))
    if name == "critical":
        assert sum(s["crit_events"] for s in sa) > 0


@pytest.mark.parametrize("name", ["leapback", "leapback_asym"])
def test_large_contexts_that_leap_back(name):
    _, after_back = _compare(_large(name), (1,) * 25 + (6,), lambda ctx, n: ctx.iterate(n))
    assert after_back > 0  # some call ended right after a leap-back


@pytest.mark.parametrize("name", ["mesh", "asym", "critical", "uneven", "general"])
def test_small_contexts_with_a_launch_per_pass(name):
    _compare(_small(name), (1, 4, 2, 5), lambda ctx, n: ctx.profile(n))


def test_small_contexts_that_leap_back():
    _, after_back = _compare(_small("leapback"), (1,) * 150, lambda ctx, n: ctx.profile(n))
    assert after_back > 0


def test_both_ways_of_stepping_in_turn():
    """One block, then launches, then one block again, poisoned between them."""
    _compare(_small("mesh"), (2, 3, 1, 4), lambda ctx, n: (ctx.iterate if n % 2 else ctx.profile)(n))


def test_the_one_block_kernels_workspace():
    """33 species on 400 subvolumes: its arrays lie outside LDS."""
    t = W.cubic_grid(20, 5, 4, periodic=False)
    _compare((_chain(33), [t] * 2, [W.poisson_state(33, t["N"], 30.0, 9 + i) for i in range(2)], 0.05, 10),
             (3, 4, 2), lambda ctx, n: ctx.iterate(n))


def test_a_lower_end_with_many_links():
    """A subvolume with 2^19 + 69 higher neighbours, more than a tile of the
    edge-parallel leap takes: the per-subvolume leap of a network of one species."""
    N = (1 << 19) + 70
    hub, leaf = np.zeros(N - 1, dtype=np.int64), np.arange(1, N, dtype=np.int64)
    topo = W.csr_from_edges(N, np.concatenate([hub, leaf]), np.concatenate([leaf, hub]), np.ones(2 * (N - 1)))
    net = W.network(["A"], [({"A": 1}, {"A": 1})], [0.0], [0.5])
    x0 = W.uniform_state(N, 500, 900, 3)
    x0[0] = 400_000_000
    _compare((net, [topo], [x0], 0.5, 10), (1, 1), lambda ctx, n: ctx.iterate(n))
