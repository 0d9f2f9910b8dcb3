"""Small realizations step inside one block each (resident_kernel), larger
ones with a launch per pass.  The same contexts through both -- plain stepping
of a context that evaluates the leap condition (theta > 0) keeps the launches
-- must agree bit for bit: counts, clock, statistics and the count of tiles
beyond a wavefront's queue; and with the oracle."""
import numpy as np
import pytest

from oracle import ffi
from pliscuda_amd import capi
from pliscuda_amd import workloads as W
from tests import helpers as H

pytestmark = pytest.mark.gpu


def _chain(S, C=1):
    """S species in a cycle of conversions and bindings, every third diffuses."""
    sp = [f"X{i}" for i in range(S)]
    rx = [({sp[i]: 1}, {sp[(i + 1) % S]: 1}) for i in range(S)] + [({sp[0]: 1, sp[1]: 1}, {sp[2]: 1}), ({}, {sp[0]: 2})]
    k = [[0.4 / (c + 1)] * S + [2e-3, 3.0] for c in range(C)]
    d = [[0.5 * (c + 1) if i % 3 == 0 else 0.0 for i in range(S)] for c in range(C)]
    return W.network(sp, rx, k, d, n_compartments=C)


def _grid(nx, ny, nz, periodic=False, comp=False):
    t = dict(W.cubic_grid(nx, ny, nz, periodic=periodic))
    if comp:
        t["comp"] = (np.arange(t["N"]) % 3 == 0).astype(np.int32)
    return t


def _case(name):
    """(network, topologies, counts, epsilon)"""
    abc = W.abc_network()
    if name.startswith("abc_"):  # edges of tiles
        t = _grid(int(name[4:]), 1, 1)
        return abc, [t], [W.poisson_state(3, t["N"], 40.0, 3)], 0.03
    if name == "uneven":
        ts = [_grid(n, n, 2) for n in (1, 3, 8, 5)]
        return abc, ts, [W.poisson_state(3, t["N"], 30.0, i) for i, t in enumerate(ts)], 0.03
    if name == "low":
        net, t, x = H.low_count_case()
        return net, [t], [x], 0.03
    if name == "leapback":
        # oversized leaps at low counts (run with n_c = 2)
        net, t, x = H.low_count_case(seed=23)
        return net, [t], [x], 0.9
    if name == "compartments":
        net, t, x = H.two_compartment_case()
        return net, [t], [x], 0.03
    if name == "asymmetric":
        t = H.asym_topology(90, 4)
        return abc, [t], [W.poisson_state(3, 90, 30.0, 5)], 0.03
    if name == "mixed":  # symmetric, weighted, asymmetric and symmetric again in one context
        ts = [_grid(5, 4, 2), W.random_mesh(4, 4, 4, 3), H.asym_topology(70, 2), _grid(4, 4, 4)]
        return abc, ts, [W.poisson_state(3, t["N"], 30.0, 5 + i) for i, t in enumerate(ts)], 0.03
    if name == "order3":
        net, t, x = H.third_order_case()
        return net, [t], [x], 0.03
    if name == "mesh":
        net, t, x = H.small_bruss()
        return net, [t], [x], 0.03
    if name == "large_means":
        net = W.network(["X"], [({}, {"X": 1}), ({"X": 1}, {})], [5000.0, 5.0], [0.1])
        t = _grid(8, 8, 5, periodic=True)
        return net, [t], [W.poisson_state(1, t["N"], 1000.0, 5)], 0.3
    if name == "dense":
        net = W.schlogl_network()
        t = _grid(9, 8, 7, periodic=True)
        return net, [t], [W.uniform_state(t["N"], 500, 600, 4)], 0.3
    if name == "no_reactions":
        net = W.network(["A", "B"], [], [], [1.0, 2.0])
        t = _grid(7, 5, 3)
        return net, [t], [W.poisson_state(2, t["N"], 20.0, 1)], 0.03
    if name == "topology_outside_lds":
        t = _grid(17, 8, 6)
        return abc, [t], [W.poisson_state(3, t["N"], 50.0, 6)], 0.03
    if name == "many_species":
        t = _grid(19, 2, 2)
        return _chain(20), [t], [W.poisson_state(20, t["N"], 30.0, 7)], 0.03
    if name == "many_species_compartments":
        t = _grid(70, 1, 1, comp=True)
        return _chain(33, 2), [t], [W.poisson_state(33, t["N"], 30.0, 8)], 0.05
    if name == "arrays_outside_lds":
        t = _grid(20, 5, 4, comp=True)
        return _chain(33, 2), [t], [W.poisson_state(33, t["N"], 30.0, 9)], 0.05
    raise KeyError(name)


CASES = ["abc_1", "abc_2", "abc_63", "abc_64", "abc_65", "abc_129", "uneven", "low", "leapback", "compartments",
         "asymmetric", "mixed", "order3", "mesh", "large_means", "dense", "no_reactions", "topology_outside_lds", "many_species",
         "many_species_compartments", "arrays_outside_lds"]


@pytest.mark.parametrize("name", CASES)
def test_resident_equals_launch_per_pass_and_oracle(name):
    net, topos, xs, eps = _case(name)
    steps, seed, nc = (200, 21, 2) if name == "leapback" else (40, 21, 10)
    ctx = capi.Context(net, topos, xs, eps=eps, nc=nc, seed=seed)
    ref = capi.Context(net, topos, xs, eps=eps, nc=nc, seed=seed)
    ref.set_tau_mode(False, theta=1.0)
    ctx.run(np.inf, step_limit=3)       # calls split differently on the two sides
    ctx.iterate(5)                      # (paused realizations stay as they are)
    ctx.run(np.inf, step_limit=steps)
    ref.run(np.inf, step_limit=steps)
    assert ctx.redo_tiles() == ref.redo_tiles()
    back = 0
    for r, t in enumerate(topos):
        a, b = ctx.stats(r), ref.stats(r)
        for f in ("t", "tau", "steps", "leapbacks", "firings", "subvolume_leaps", "crit_events", "status"):
            assert a[f] == b[f], (r, f, a[f], b[f])
        assert np.array_equal(ctx.get_state(r), ref.get_state(r))
        x = np.array(xs[r], dtype=np.uint32).copy()
        so = ffi.run(ffi.Model(net, t), x, eps, nc, seed, np.inf, step_limit=steps, realization=r)
        assert np.array_equal(ctx.get_state(r), x) and a["t"] == so.t and a["firings"] == so.firings
        back += a["leapbacks"]
    assert back > 0 if name == "leapback" else True
    ctx.close()
    ref.close()


def test_resident_clamps_pauses_absorbs_and_resumes():
    """t_end and t_pause, a realization with no event left, and a checkpoint
    taken between calls, against the launch-per-pass step."""
    net = W.network(["A"], [({"A": 1}, {})], [2.0], [0.3])
    topos = [_grid(4, 4, 1), _grid(5, 1, 1)]
    xs = [W.poisson_state(1, 16, 60.0, 1), np.zeros(5, dtype=np.uint32)]
    out = []
    for theta in (0.0, 1.0):
        ctx = capi.Context(net, topos, xs, seed=9)
        ctx.set_tau_mode(False, theta=theta)
        ctx.run(2.0, t_pause=0.1)
        blob = ctx.checkpoint()
        got = [(ctx.get_state(r), ctx.stats(r)) for r in range(2)]
        ctx.run(0.5)
        ctx.restore(blob)
        ctx.run(0.5)
        got += [(ctx.get_state(r), ctx.stats(r)) for r in range(2)]
        ctx.run(40.0)  # everything has decayed
        got += [(ctx.get_state(r), ctx.stats(r)) for r in range(2)]
        out.append(got)
        ctx.close()
    for (xa, sa), (xb, sb) in zip(*out):
        assert np.array_equal(xa, xb)
        for f in ("t", "tau", "steps", "leapbacks", "firings", "crit_events", "status"):
            assert sa[f] == sb[f], f
    assert out[0][-2][1]["status"] == 2 and out[0][2][1]["t"] == 0.5
