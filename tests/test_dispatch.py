"""The rules that choose a context's way of stepping (plis_dispatch.h), on the CPU:
compiled by themselves and asked for sizes whose two sides were measured."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "pliscuda_amd", "csrc")

MAIN = r"""
#include <cstdio>
#include "plis_dispatch.h"
using namespace plis;
// S R general count blocks_per_cu {N n_in}...: realizations of the given sizes in turn
int main() {
    int S, R, general;
    unsigned long count, per_cu, kinds;
    while (std::scanf("%d %d %d %lu %lu %lu", &S, &R, &general, &count, &per_cu, &kinds) == 6) {
        std::vector<StepSize> k(kinds), rs;
        for (auto& r : k) {
            unsigned long N, E;
            if (std::scanf("%lu %lu", &N, &E) != 2) return 1;
            r = {N, E, (N + 63) / 64};
        }
        for (unsigned long i = 0; i < count; ++i) rs.push_back(k[i % kinds]);
        const double us = resident_step_us(S, R, rs, 256 * per_cu);
        std::printf("%d %.3f %u\n", (int)resident_pays(S, R, general != 0, rs, 256 * per_cu), us, resident_launch_iters(us));
    }
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("dispatch")
    (d / "main.cpp").write_text(MAIN)
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, str(d / "main.cpp"), "-o", str(d / "rule")],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr

    def ask(S, R, general, count, per_cu, *sizes):
        line = " ".join(str(v) for v in (S, R, int(general), count, per_cu, len(sizes))) + " "
        out = subprocess.run([str(d / "rule")], input=line + " ".join(f"{n} {e}" for n, e in sizes), capture_output=True,
                             text=True, check=True).stdout.split()
        return out[0] == "1", float(out[1]), int(out[2])

    return ask


# (S, R, (N, in-edges), blocks a CU, realizations, one block each): 1 where that was the faster side by 5 % or more, 0
# where the launches were
MEASURED = [
    (3, 3, (64, 288), 4, 1, 1), (3, 3, (64, 288), 4, 3000, 1),
    (3, 3, (216, 1080), 1, 256, 1), (3, 3, (216, 1080), 1, 257, 1), (3, 3, (216, 1080), 1, 3000, 0),
    (3, 3, (729, 3888), 1, 256, 1), (3, 3, (729, 3888), 1, 512, 1), (3, 3, (1000, 5400), 1, 1, 0),
    (1, 4, (125, 750), 2, 512, 1), (1, 4, (125, 750), 2, 2048, 0), (1, 4, (125, 750), 2, 4096, 0),
    (1, 4, (216, 1296), 1, 512, 1), (1, 4, (216, 1296), 1, 1024, 0), (1, 4, (216, 1296), 1, 3000, 0),
    (1, 4, (512, 3072), 1, 257, 0), (1, 4, (512, 3072), 1, 512, 1), (1, 4, (729, 4374), 1, 257, 0),
    (1, 1, (64, 288), 4, 4096, 1), (1, 1, (216, 1080), 1, 3000, 0), (1, 1, (125, 600), 2, 4096, 0),
    (1, 1, (512, 2688), 1, 1024, 1), (1, 1, (1728, 9504), 1, 1, 0),
    (5, 8, (64, 482), 2, 768, 1), (5, 8, (64, 482), 2, 4096, 0), (5, 8, (216, 1718), 1, 1024, 1),
    (5, 8, (216, 1718), 1, 3000, 0),
    (8, 12, (64, 288), 1, 1024, 1), (8, 12, (64, 288), 1, 2048, 0), (8, 12, (343, 1764), 1, 768, 1),
]


@pytest.mark.parametrize("S,R,size,per_cu,count,one_block", MEASURED)
def test_the_faster_side_is_chosen(rule, S, R, size, per_cu, count, one_block):
    assert rule(S, R, False, count, per_cu, size)[0] == bool(one_block)


def test_the_general_instantiation_stays_with_one_block(rule):
    for count in (1, 256, 4096):
        assert rule(32, 62, True, count, 1, (60, 118))[0]


def test_uneven_realizations_are_scheduled_one_after_the_other(rule):
    """A few large realizations among many small ones: a large one starts at the
    latest when the first small one has ended, so the step lasts no longer than
    the two together, not two rounds of the large one."""
    large, small = rule(3, 3, False, 1, 1, (700, 3700))[1], rule(3, 3, False, 1, 1, (8, 24))[1]
    pays, us, _ = rule(3, 3, False, 320, 1, (700, 3700), *[(8, 24)] * 9)
    assert pays and us == pytest.approx(large + small, rel=1e-3) and us < 1.5 * large
    assert rule(3, 3, False, 256, 1, (700, 3700))[1] == pytest.approx(large, rel=1e-3)
    assert rule(3, 3, False, 257, 1, (700, 3700))[1] == pytest.approx(2 * large, rel=1e-3)


@pytest.mark.parametrize("S,R,general,size,count", [
    (1, 1, False, (1, 0), 1), (3, 3, False, (64, 288), 1), (3, 3, False, (900, 4900), 256), (32, 62, True, (60, 118), 1),
    (32, 62, True, (60, 118), 65536), (32, 62, True, (2600, 5198), 1), (64, 128, True, (1200, 2398), 5000)])
def test_a_launch_of_one_block_kernels_is_short(rule, S, R, general, size, count):
    """About 50 ms however large the network and however many the realizations, and
    no shorter than it has to be."""
    pays, us, iters = rule(S, R, general, count, 1, size)
    assert pays and 1 <= iters <= 1024
    assert iters == 1 or iters * us <= 50e3
    assert iters == 1024 or (iters + 1) * us > 50e3


@pytest.mark.gpu
def test_a_call_of_several_launches():
    """38 species, 40 reactions on 900 subvolumes: a launch makes some 480 iterations.
    One call of 700 equals a launch per pass, which evaluates the leap condition."""
    from pliscuda_amd import capi
    from pliscuda_amd import workloads as W

    S = 38
    sp = [f"X{i}" for i in range(S)]
    rx = [({sp[i]: 1}, {sp[(i + 1) % S]: 1}) for i in range(S)] + [({sp[0]: 1, sp[1]: 1}, {sp[2]: 1}), ({}, {sp[0]: 2})]
    net = W.network(sp, rx, [0.4] * S + [2e-3, 3.0], [0.5 if i % 3 == 0 else 0.0 for i in range(S)])
    topo = W.cubic_grid(900, 1, 1, periodic=False)
    x0 = W.poisson_state(S, 900, 30.0, 7)
    out = []
    for theta in (0.0, 1.0):
        ctx = capi.Context(net, [topo], [x0], seed=4)
        ctx.set_tau_mode(False, theta=theta)
        ctx.arm(step_limit=700)
        ctx.iterate(700)
        out.append((ctx.get_state(0), ctx.stats(0)))
        ctx.close()
    (xa, sa), (xb, sb) = out
    assert np.array_equal(xa, xb) and all(sa[f] == sb[f] for f in ("t", "steps", "leapbacks", "firings", "crit_events"))
    assert sa["steps"] + sa["leapbacks"] == 700
