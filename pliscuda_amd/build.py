"""Builds libplis_hip.so (gfx950) and the ``pliscuda`` driver in-tree.

    python -m pliscuda_amd.build
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libplis_hip.so")
BIN_DIR = os.path.join(HERE, "bin")
DRIVER = os.path.join(BIN_DIR, "pliscuda")

# -ffp-contract=off: the kernels spell out every fused multiply-add, so the
# host oracle can execute the same IEEE operations.  Packed FP32 is disabled.
HIP_FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
             "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def _run(cmd):
    print("+", " ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)


# (species, reactions) bounds the step kernels are instantiated for, smallest
# fitting one is used: Schlogl-like, A-B-C, Brusselator, <= 8 x 16, general
VARIANTS = [(1, 4), (3, 4), (5, 8), (8, 16), (64, 128)]


def build_lib():
    obj = os.path.join(HERE, "_build")
    os.makedirs(obj, exist_ok=True)
    jobs = [("plis_capi", "plis_capi.hip", []), ("plis_resident", "plis_resident.hip", [])]
    for s, r in VARIANTS:
        defs = [f"-DPLIS_MS={s}", f"-DPLIS_MR={r}"]
        # without loop-invariant code motion in the back end the constants of
        # rare inner loops (inversion search, PTRS) are formed there instead of
        # held in registers over the whole kernel: phase_b_kernel 109 -> 73 us,
        # phase_a_kernel 72.8 -> 68.6 us on the 1M-subvolume Brusselator mesh
        jobs.append((f"plis_variant_{s}_{r}", "plis_variant.hip", [*defs, "-mllvm", "-disable-machine-licm"]))
        if s <= 8:
            jobs.append((f"plis_variant_learned_{s}_{r}", "plis_variant_learned.hip",
                         [*defs, "-mllvm", "-disable-machine-licm"]))

    def compile_one(job):
        name, src, defs = job
        out = os.path.join(obj, name + ".o")
        _run(["hipcc", *HIP_FLAGS, *defs, "-c", "-o", out, os.path.join(CSRC, src)])
        return out

    # the largest first: the build lasts as long as it does
    with ThreadPoolExecutor(max_workers=min(8, os.cpu_count() or 1)) as pool:
        objs = list(pool.map(compile_one, reversed(jobs)))
    _run(["hipcc", "--offload-arch=gfx950", "-shared", "-o", LIB + ".tmp", *objs])
    os.replace(LIB + ".tmp", LIB)


def build_driver():
    os.makedirs(BIN_DIR, exist_ok=True)
    host = os.path.join(CSRC, "host")
    srcs = [os.path.join(host, f) for f in ("plis_inputs.cpp", "driver.cpp", "main.cpp")]
    _run(["g++", "-std=c++17", "-O2", "-Wall", "-I", os.path.join(ROOT, "include"), "-I", host,
          "-o", DRIVER + ".tmp", *srcs, "-L", HERE, "-lplis_hip", f"-Wl,-rpath,$ORIGIN/.."])
    os.replace(DRIVER + ".tmp", DRIVER)


def build_all():
    build_lib()
    if os.path.exists(os.path.join(CSRC, "host", "main.cpp")):
        build_driver()


if __name__ == "__main__":
    build_all()
    sys.exit(0)
