"""The pointer to a kernel's arguments is taken in kernels only.

The compiler's builtin for it gives null in any other function, which goes
unseen as long as all of them are inlined into their kernel: a change of
inlining would turn path recording into accesses near address 0. Checked in the
device code before inlining."""
import os
import re
import shutil
import subprocess

import pytest

from robast_amd import build as B


def test_argument_pointer_is_taken_in_kernels(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    ir = str(tmp_path / "rbgpu.ll")
    subprocess.check_call([hipcc, "--offload-arch=gfx950", "-O1", "-std=c++17", "-ffp-contract=off", "-w", "-Xclang",
                           "-disable-llvm-passes", "--cuda-device-only", "-S", "-emit-llvm", "-o", ir, B.SRC])
    kernels = others = 0
    inside = ""
    with open(ir) as f:
        for line in f:
            if line.startswith("define"):
                inside = line
            elif re.search(r"call .*@llvm\.amdgcn\.kernarg\.segment\.ptr", line):
                if " amdgpu_kernel " in inside:
                    kernels += 1
                else:
                    others += 1
    assert kernels > 0 and others == 0, (kernels, others)
