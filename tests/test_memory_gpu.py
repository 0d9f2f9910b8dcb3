"""A device that is nearly full: a context that has no room for the edge-parallel
leap's buffers is made without them and steps the same trajectory.  (Up to 8
species: the general step kernels need 1.4 GB of scratch memory themselves.)"""
import ctypes as C

import numpy as np
import pytest

from oracle import ffi
from pliscuda_amd import capi
from pliscuda_amd import workloads as W
from tests import helpers as H
from tests.test_launched_gpu import _directed

pytestmark = pytest.mark.gpu


class _Filled:
    """Holds all of the device's memory but `leave` bytes."""

    def __init__(self, leave):
        self.hip = C.CDLL("libamdhip64.so")
        self.hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
        self.hip.hipFree.argtypes = [C.c_void_p]
        self.leave, self.held = leave, []

    def free(self):
        a, b = C.c_size_t(), C.c_size_t()
        assert self.hip.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    def __enter__(self):
        for _ in range(64):  # (a device may not give all of it in one piece)
            want = min(self.free() - self.leave, 32 << 30)
            if want < 16 << 20:
                return self
            p = C.c_void_p()
            if self.hip.hipMalloc(C.byref(p), want) != 0:
                break
            self.held.append(p)
        self.__exit__()
        pytest.skip("the device's memory could not be filled to the size wanted")

    def __exit__(self, *_):
        for p in self.held:
            self.hip.hipFree(p)
        self.held = []


def _warm():
    """(Allocations that outlast a context are made.)"""
    t = W.cubic_grid(4, 4, 4, periodic=False)
    with capi.Context(W.abc_network(), [t], [W.poisson_state(3, 64, 50.0, 5)]) as ctx:
        ctx.run(np.inf, step_limit=3)


def _case(kind):
    """160,380 subvolumes: the large buffers would take some 15 MiB."""
    net, topo = W.abc_network(), dict(W.cubic_grid(55, 54, 54, periodic=False))
    if kind == "asym":
        topo = _directed(topo, True)
    elif kind == "compartments":
        net = H.two_compartment_case()[0]
        topo["comp"] = (np.arange(topo["N"]) % 3 == 0).astype(np.int32)
    return net, topo, W.poisson_state(3, topo["N"], [40.0, 12.0, 30.0], 8)


KINDS = ["grid", "asym", "compartments"]
STEPS = 9


@pytest.fixture(scope="module")
def made():
    """768 MiB left, less than the 1 GiB that a context of this size leaves free.  One
    of 64 subvolumes takes a negligible part of it and keeps its buffers."""
    _warm()
    out = {}
    with _Filled(768 << 20):
        t = W.cubic_grid(4, 4, 4, periodic=False)
        with capi.Context(W.abc_network(), [t], [W.poisson_state(3, 64, 50.0, 5)]) as ctx:
            ctx.arm()
            out["box"] = ctx.profile_kernels(1)[7]
        for kind in KINDS:
            net, topo, x0 = _case(kind)
            ctx = capi.Context(net, [topo], [x0], eps=0.1, seed=9)
            ctx.run(np.inf, step_limit=STEPS - 5)
            blob = ctx.checkpoint()
            ctx.arm(step_limit=STEPS - 3)
            completion = ctx.profile_kernels(1)[7]
            ctx.debug_poison()
            ctx.run(np.inf, step_limit=STEPS)
            out[kind] = ctx.get_state(0), ctx.stats(0), blob, completion
            ctx.close()
    return out


@pytest.mark.parametrize("kind", KINDS)
def test_a_context_without_room_for_the_large_buffers(made, kind):
    """The per-subvolume leap, which has no kernel of its own to complete it, gives
    the oracle's trajectory; a checkpoint goes on in a context that has room."""
    net, topo, x0 = _case(kind)
    x, st, blob, completion = made[kind]
    assert completion == 0.0 and made["box"] > 0.0
    xo = np.array(x0, dtype=np.uint32).copy()
    so = ffi.run(ffi.Model(net, topo), xo, 0.1, 10, 9, np.inf, step_limit=STEPS)
    assert np.array_equal(x, xo)
    for f in ("steps", "leapbacks", "firings", "crit_events", "t", "status"):
        assert st[f] == getattr(so, f), f
    ctx = capi.Context(net, [topo], [x0], eps=0.1, seed=9)
    ctx.restore(blob)
    ctx.run(np.inf, step_limit=STEPS)
    assert np.array_equal(ctx.get_state(0), xo)
    ctx.close()
