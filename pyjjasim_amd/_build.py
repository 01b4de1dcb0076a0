"""Build libjja.so in-tree with hipcc for gfx950.

The shared library holds the HIP kernels, the device plan and the host-side
Cholesky factorisation. It is built next to this file so that it travels with the
source tree; nothing is installed elsewhere. The sources compile side by side
(each to an object in a temporary folder) and are linked once.
"""
import os
import subprocess
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libjja.so")

HIPCC_FLAGS = [
    "-O3", "--offload-arch=gfx950", "-fPIC", "-std=c++17",
    # the step expressions keep the reference's operation order: no FMA contraction
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # invariants of the step loop stay where they are used: hoisted, they spill in the
    # kernels that keep phases in registers; the general kernels do not mind (us a step with
    # and without hoisting: 512x512, 16 columns 284.9 / 275.8, 100x100 in 4 parts with the
    # factor 179.4 / 173.9, 60x60 triangular with stencil 4 300.1 / 298.2; 52 runs of small
    # circuits 0.98 to 1.05 times as fast without)
    "-Wall", "-Wno-unused-result", "-mllvm", "-disable-machine-licm",
]


def sources():
    return [os.path.join(CSRC, name) for name in ("jja_evolve.hip", "jja_resident.hip", "jja_slab.hip", "jja_wide.hip", "jja_domain.hip", "jja_factor.cpp", "jja_program.cpp")]


def build_library(verbose=False):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

    def run(cmd):
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.run(cmd, check=True)

    with tempfile.TemporaryDirectory() as tmp:
        objects = [os.path.join(tmp, os.path.basename(src) + ".o") for src in sources()]
        with ThreadPoolExecutor(len(objects)) as pool:
            list(pool.map(lambda so: run([hipcc, *HIPCC_FLAGS, "-c", so[0], "-o", so[1]]), zip(sources(), objects)))
        out = LIB + ".tmp"
        run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *objects, "-o", out])
    os.replace(out, LIB)
    return LIB


if __name__ == "__main__":
    print(build_library(verbose=True))
