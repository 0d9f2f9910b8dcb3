"""Draws made at once inside the leap's walk (dense tiles) against the oracle, bit
for bit: hop means from below one to beyond the squeeze's range, ragged tiles,
compartments and asymmetric weights; and the squeeze as the kernels form it."""
import numpy as np
import pytest

from oracle import ffi
from pliscuda_amd import capi
from pliscuda_amd import workloads as W
from tests import helpers as H


def _case(kind, count):
    if kind == "asym":
        net, topo = W.abc_network(), H.asym_topology(2001, 3)
    elif kind == "comp":
        net = H.two_compartment_case()[0]
        topo = dict(W.cubic_grid(13, 13, 11, periodic=False))
        topo["comp"] = (np.arange(topo["N"]) % 3 == 0).astype(np.int32)
    elif kind == "one":
        net = W.network(["A"], [({"A": 1}, {}), ({}, {"A": 1})], [0.1, 0.1 * count], [5.0])
        topo = W.cubic_grid(13, 11, 15, periodic=False)
    else:
        net, topo = W.schlogl_network(), W.cubic_grid(17, 11, 13, periodic=True)
    means = [count] * net["S"]
    return net, topo, W.poisson_state(net["S"], topo["N"], means, 8)


CASES = [(k, c) for k in ("one", "schlogl", "asym", "comp") for c in (40, 200, 700, 4000)]


@pytest.mark.gpu
@pytest.mark.parametrize("kind,count", CASES)
def test_dense_draws(kind, count):
    net, topo, x0 = _case(kind, count)
    eps, nc, seed, steps = 0.2, 10, 6, 12
    ctx = capi.Context(net, [topo], [x0], eps=eps, nc=nc, seed=seed)
    ctx.run(np.inf, step_limit=steps)
    x = np.array(x0, dtype=np.uint32).copy()
    st = ffi.run(ffi.Model(net, topo), x, eps, nc, seed, np.inf, step_limit=steps)
    g, gs = ctx.get_state(0), ctx.stats(0)
    ctx.close()
    assert np.array_equal(g, x)
    for f in ("steps", "leapbacks", "firings", "crit_events", "t", "status"):
        assert gs[f] == getattr(st, f), f


def _squeeze(l, u):
    """The kernels' squeeze in single precision (u -+ delta against G)."""
    f = np.float32
    n = np.rint(f(l * f(1.44269502)))
    r = np.float32(np.float64(n) * float.fromhex("0x1.62e4p-1") - np.float64(l))  # exact product, one rounding
    r = np.float32(np.float64(n) * float.fromhex("0x1.7f7d1cp-20") + np.float64(r))
    p = f(float.fromhex("0x1.a01a02p-13"))
    for c in ("0x1.6c16c2p-10", "0x1.111112p-7", "0x1.555556p-5", "0x1.555556p-3", "0x1p-1", "0x1p+0", "0x1p+0"):
        p = np.float32(np.float64(p) * np.float64(r) + float.fromhex(c))
    p = f(p * f(2.0 ** -int(n)))
    G, lo, hi, k = p, f(u - f(2.0 ** -15)), f(u + f(2.0 ** -15)), 0
    for j in range(1, 16):
        if not G < lo:
            break
        p = f(f(p * l) * f(1.0 / j))
        G = f(G + p)
        k = j
    return k if G >= hi else -1


@pytest.mark.parametrize("lam", [1e-3, 0.3, 1.0, 2.5, 6.0, 9.989])
def test_squeeze_form_decides_as_the_double_search(lam):
    """What it decides is the double search's result, also for uniforms at a
    cumulative probability's edge and for a mean off by 8 2^-24; those within
    delta (and few others) it leaves open."""
    rng = np.random.Generator(np.random.PCG64(5))
    pk, F, edges = np.exp(-lam), np.exp(-lam), []
    for k in range(1, 16):
        edges.append(F)
        pk *= lam / k
        F += pk
    us = list(rng.random(300))
    for e in edges:
        us += [e + s * d for s in (-1, 1) for d in (2.0 ** -20, 2.0 ** -16, 3.5e-5, 4.5e-5, 1e-4)]
    left = 0
    for u in us:
        w = min(max(int(u * 2.0 ** 32), 0), 2 ** 32 - 1)
        ud = (w + 0.5) * 2.0 ** -32
        p = F = np.exp(-lam)
        exact = 0
        while ud > F and exact < 1000:
            exact += 1
            p = p * lam / exact
            F += p
        for off in (-1, 0, 1):
            k = _squeeze(np.float32(lam * (1 + off * 8 * 2.0 ** -24)), np.float32(np.float32(w) * np.float32(2.0 ** -32)))
            assert k in (-1, exact), (u, off, k, exact)
            left += k < 0 and min([abs(ud - e) for e in edges] or [1.0]) > 1e-4 and exact <= 15
    assert left == 0
