"""Builds librbgpu.so in-tree: hipcc for gfx950, packed-FP32 instructions
disabled (-packed-fp32-ops), and no contraction of separate multiplies and
adds into FMAs (-ffp-contract=off): every FP64 operation then rounds as
written, as in the CPU oracle, which makes the Davies-Cotton trace
bit-identical to it for a 1 % longer kernel.

Machine-level loop-invariant code motion is off: it hoists the literals of the
FP64 code out of the tracing loops into registers those loops do not have
(Davies-Cotton trace kernel at 1e7 rays 3.20 ms without it, 3.84 with it;
alignment gradient kernel 4.60 and 5.20). The other kernels, whole traces in
us without it and with it: persistent schedule 1e6 rays 1199 and 1215, mixed
3e5 355 and 354, two levels deep 2e5 481 and 530, deep mixed 1e6 1203 and 1400,
a lens 1e6 1199 and 1212, mixed gradient 8e5 808 and 810, light guides 1e6 equal
within their spread; unsorted rough facets lose (2e4 247 and 230, 2e5 473 and
463; the unrolled sphere code gives most of it back)."""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "csrc", "rbgpu.hip")
OUT = os.path.join(HERE, "librbgpu.so")

FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-ffp-contract=off", "-mllvm", "-disable-machine-licm=1", "-Wno-unused-result"]


def build(verbose=False):
    cmd = ["/opt/rocm/bin/hipcc", *FLAGS, "-o", OUT + ".tmp", SRC]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    os.replace(OUT + ".tmp", OUT)
    return OUT


if __name__ == "__main__":
    build(verbose="-v" in sys.argv)
