"""How many iterations a run launches at once: one that may end at any step, since
nothing can happen any more, must not pay for a long batch of empty ones."""
import time

import numpy as np
import pytest

from pliscuda_amd import capi
from pliscuda_amd import workloads as W

pytestmark = pytest.mark.gpu


def _elapsed(f):
    t = time.perf_counter()
    f()
    return time.perf_counter() - t


def test_a_run_that_is_absorbed_early_launches_few_empty_iterations():
    """Three molecules decay on 8,000 subvolumes (a launch per pass).  The run may
    launch as many iterations again as it made steps, here well below 64; 256
    finished iterations in one call are the measure of what more would cost."""
    net = W.network(["A"], [({"A": 1}, {})], [2.0], [0.3])
    topo = W.cubic_grid(20, 20, 20, periodic=False)
    x0 = np.zeros(topo["N"], dtype=np.uint32)
    x0[5] = 3
    run, idle = [], []
    for _ in range(4):
        ctx = capi.Context(net, [topo], [x0], seed=9)
        ctx.run(np.inf, step_limit=1)  # graphs are captured
        run.append(_elapsed(lambda: ctx.run(np.inf)))
        st = ctx.stats(0)
        assert st["status"] == 2 and st["steps"] < 32

        def empty():
            ctx.iterate(256)
            ctx.sync()

        idle.append(_elapsed(empty))
        assert ctx.stats(0)["steps"] == st["steps"]
        ctx.close()
    assert min(run) < 0.6 * min(idle), (run, idle)


def test_a_source_in_one_of_two_compartments_still_absorbs():
    """Only the second compartment has a source, so a realization that lies in the
    first can be absorbed, and is."""
    net = W.network(["A"], [({"A": 1}, {}), ({}, {"A": 1})], [[2.0, 0.0], [2.0, 50.0]], [[0.3], [0.3]], n_compartments=2)
    out = []
    for comp in (0, 1):
        topo = dict(W.cubic_grid(12, 12, 12, periodic=False))
        topo["comp"] = np.full(topo["N"], comp, dtype=np.int32)
        x0 = np.zeros(topo["N"], dtype=np.uint32)
        x0[7] = 2
        ctx = capi.Context(net, [topo], [x0], seed=3)
        ctx.run(np.inf, step_limit=100)
        out.append(ctx.stats(0))
        ctx.close()
    assert out[0]["status"] == 2 and out[0]["steps"] < 100
    assert out[1]["status"] == 1 and out[1]["steps"] == 100
