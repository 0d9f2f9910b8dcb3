"""Stepping with a launch per pass at sizes and in forms that no other test has:
tiles of one wavefront each (more than 1,024) with compartments and asymmetric
weights, calls that end after leap-backs, checkpoints, runs without graphs, and
learned and judged contexts on topologies that are not symmetric."""
import numpy as np
import pytest

from oracle import ffi
from pliscuda_amd import capi, learned
from pliscuda_amd import workloads as W
from tests import helpers as H
from tests.test_draw_tiers_launched_gpu import _many

pytestmark = pytest.mark.gpu

FIELDS = ("steps", "leapbacks", "firings", "crit_events", "t", "status")


def _directed(t, cut):
    """Weights that differ by direction; cut: every 97th link loses its way back."""
    src = np.repeat(np.arange(t["N"], dtype=np.int64), np.diff(t["row_ptr"].astype(np.int64)))
    dst = t["col"].astype(np.int64)
    w = np.where(dst > src, 1.25, 0.5)
    keep = ~((src > dst) & (src % 97 == 5)) if cut else np.ones(len(src), dtype=bool)
    return W.csr_from_edges(t["N"], src[keep], dst[keep], w[keep])


def _topology(kind, sides):
    t = dict(W.cubic_grid(*sides, periodic=False))
    if "asym" in kind:
        t = _directed(t, True)
    if "compartments" in kind:
        t["comp"] = (np.arange(t["N"]) // 7 % 2).astype(np.int32)
    return t


def _network(S, kind):
    if S == 3:
        return H.two_compartment_case()[0] if "compartments" in kind else W.abc_network()
    if S == 1:
        C = 2 if "compartments" in kind else 1
        return W.network(["A"], [({}, {"A": 1}), ({"A": 1}, {})], [[20.0 / (c + 1), 0.5] for c in range(C)],
                         [[2.0 / (c + 1)] for c in range(C)], n_compartments=C)
    if S == 5:
        b = W.brusselator_network(W.SEED_BRUSS)
        if "compartments" not in kind:
            return b
        return dict(b, C=2, k=np.concatenate([np.ravel(b["k"]), 0.5 * np.ravel(b["k"])]).reshape(2, -1),
                    d=np.concatenate([np.ravel(b["d"]), 2.0 * np.ravel(b["d"])]).reshape(2, -1))
    return _many(S, 16, 2 if "compartments" in kind else 1)


def _matches(ctx, net, topo, x0, eps, nc, seed, real=0):
    x, st = np.array(x0, dtype=np.uint32).copy(), ctx.stats(real)
    so = ffi.run(ffi.Model(net, topo), x, eps, nc, seed, np.inf, step_limit=st["steps"], realization=real)
    assert np.array_equal(ctx.get_state(real), x)
    for f in ("steps", "firings", "t"):
        assert st[f] == getattr(so, f), f


@pytest.mark.parametrize("kind", ["asym", "compartments", "asym_compartments"])
@pytest.mark.parametrize("S,shape", [(s, (0, 0)) for s in (1, 3, 5, 8)] + [(s, sh) for s in (3, 5) for sh in ((1, 3), (4, 2))])
def test_a_wavefront_per_tile(S, kind, shape):
    """41 x 41 x 40 subvolumes are 1,051 tiles, the last one ragged: up to 3 species
    draw dense tiles in the walk, more always queue; with blocks that take one
    tile a wavefront and with few that go round."""
    net, topo = _network(S, kind), _topology(kind, (41, 41, 40))
    x0 = W.poisson_state(S, topo["N"], [400.0 if s % 2 == 0 else 15.0 for s in range(S)], 8)
    ctx = capi.Context(net, [topo], [x0], eps=0.1, seed=9, waves_per_block=shape[0], blocks_per_cu=shape[1])
    assert ctx.launch_shape()["tiles"] > 1024
    ctx.run(np.inf, step_limit=2)
    ctx.run(np.inf, step_limit=5)
    _matches(ctx, net, topo, x0, 0.1, 10, 9)
    ctx.close()


@pytest.mark.parametrize("kind,case", [(k, c) for k in ("grid", "asym", "compartments") for c in ("leapbacks", "steps")])
def test_iterations_split_into_calls(kind, case):
    """Calls of one iteration and of many, ending after accepted steps and after
    leap-backs, against one call."""
    eps, nc = (0.9, 0) if case == "leapbacks" else (0.05, 10)
    net, topo = _network(3, kind), _topology(kind, (13, 13, 11))
    x0 = W.poisson_state(3, topo["N"], [2.0, 2.0, 1.0] if case == "leapbacks" else 40.0, 8)
    calls, out, ended = (1,) * 30 + (4, 2, 9), [], 0
    for split in (False, True):
        ctx = capi.Context(net, [topo], [x0], eps=eps, nc=nc, seed=9)
        ctx.arm()
        for n in calls if split else (sum(calls),):
            before = ctx.stats(0)["leapbacks"]
            ctx.iterate(n)
            ended += split and n == 1 and ctx.stats(0)["leapbacks"] > before
        out.append((ctx.get_state(0), ctx.stats(0)))
        _matches(ctx, net, topo, x0, eps, nc, 9)
        ctx.close()
    (xa, sa), (xb, sb) = out
    assert np.array_equal(xa, xb) and all(sa[f] == sb[f] for f in FIELDS)
    assert ended > 0 or case == "steps"


@pytest.mark.parametrize("use_graph", [True, False])
def test_with_and_without_graphs(use_graph):
    net, topo = W.schlogl_network(), W.cubic_grid(13, 11, 17, periodic=True)
    x0 = W.uniform_state(topo["N"], 80, 600, 4)
    ctx = capi.Context(net, [topo], [x0], seed=9, use_graph=use_graph)
    for n in (1, 2, 30, 97):
        ctx.run(np.inf, step_limit=n)
    _matches(ctx, net, topo, x0, 0.03, 10, 9)
    ctx.close()


@pytest.mark.parametrize("kind", ["grid", "asym", "compartments"])
def test_checkpoints_at_every_point(kind):
    """Taken after an accepted step and right after a leap-back, restored into a new
    context and into the one that ran on."""
    net, topo = _network(3, kind), _topology(kind, (13, 13, 11))
    x0 = W.poisson_state(3, topo["N"], [2.0, 2.0, 1.0], 8)
    a = capi.Context(net, [topo], [x0], eps=0.9, nc=0, seed=9)
    a.arm()
    blobs = {}
    for _ in range(30):
        before = a.stats(0)["leapbacks"]
        a.iterate(1)
        after = "leap-back" if a.stats(0)["leapbacks"] > before else "step"
        if after not in blobs:
            blobs[after] = a.checkpoint()
    assert len(blobs) == 2
    for blob in blobs.values():
        got = []
        b = capi.Context(net, [topo], [np.zeros_like(x0)], eps=0.9, nc=0, seed=9)
        for ctx in (a, b):
            ctx.restore(blob)
            ctx.run(np.inf, step_limit=25)
            got.append((ctx.get_state(0), ctx.stats(0)))
        _matches(b, net, topo, x0, 0.9, 0, 9)
        b.close()
        assert np.array_equal(got[0][0], got[1][0]) and all(got[0][1][f] == got[1][1][f] for f in FIELDS)
    a.close()


@pytest.mark.parametrize("rejected", [False, True])
@pytest.mark.parametrize("kind", ["grid", "asym", "compartments", "asym_compartments"])
@pytest.mark.parametrize("S,relu", [(3, False), (5, False), (5, True), (8, False), (8, True)])
def test_learned_proposals_of_the_leap_equal_the_tau_pass(S, kind, relu, rejected):
    """The proposals made while the leap is completed equal those of the tau pass on
    the same counts, which setting the state forces before each step; the counts
    of broken leap conditions are the oracle's.  Proposals short enough to be
    kept, and long ones that the judge turns down."""
    net, topo = _network(S, kind), _topology(kind, (11, 9, 8))
    x0 = W.poisson_state(S, topo["N"], 60.0, 8)
    plain = capi.Context(net, [topo], [x0], eps=0.05, seed=5)
    plain.run(np.inf, step_limit=1)
    log_tau = np.log(plain.stats(0)["tau"])
    plain.close()
    norm = np.concatenate([np.zeros(12), np.ones(12), [log_tau + (4.0 if rejected else -2.0), 1.0]]).astype(np.float32)
    runs = []
    for force in (False, True):
        ctx = capi.Context(net, [topo], [x0], eps=0.05, seed=5)
        ctx.mlp_activation(0 if relu else 1)
        ctx.mlp_set(learned.init_weights(7), norm)
        ctx.set_tau_mode(True, kappa=1.0, theta=1.0, viol_rate_max=0.02 if rejected else 1.0)
        prev, total, model = np.array(x0, dtype=np.uint32), 0, ffi.Model(net, topo)
        for k in range(1, 16):
            ctx.run(np.inf, step_limit=k)
            if force:
                x = ctx.get_state(0)
                total += ffi.violations(model, prev, x, 0.05, 10, 1.0)[0]
                assert ctx.stats(0)["violations"] == total
                prev = x
                ctx.set_state(0, x)
        runs.append((ctx.get_state(0), ctx.stats(0)))
        ctx.close()
    (xa, sa), (xb, sb) = runs
    assert np.array_equal(xa, xb)
    for f in FIELDS + ("learned_steps", "learned_rejects", "violations"):
        assert sa[f] == sb[f], f
    assert sa["learned_rejects" if rejected else "learned_steps"] > 0


@pytest.mark.parametrize("kind", ["grid", "asym", "compartments"])
def test_a_judged_context_completes_its_leap_in_a_kernel_of_its_own(kind):
    """plis_profile_kernels reports it (its slot holds the gap between two events in
    a context that has none, so the judged one's is compared with that)."""
    net, topo = _network(5, kind), _topology(kind, (33, 32, 31))
    x0 = W.poisson_state(5, topo["N"], 60.0, 8)
    ms = []
    for theta in (0.0, 1.0):
        ctx = capi.Context(net, [topo], [x0], seed=9)
        ctx.set_tau_mode(False, theta=theta)
        ctx.arm()
        ctx.profile_kernels(2)
        ps = [ctx.profile_kernels(5) for _ in range(6)]  # (the least of several: a host that was held up adds to a gap)
        assert all(p[5] > 0.0 and p[6] == 0.0 for p in ps)
        ms.append(min(p[7] for p in ps))
        _matches(ctx, net, topo, x0, 0.03, 10, 9)
        ctx.close()
    assert ms[1] > ms[0] >= 0.0
