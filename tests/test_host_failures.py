"""A host batch whose wait for the device fails half way.

The call hands its work area and pinned memory back when it returns, for the
next call to overwrite, so no copy may still be on its way then, whichever
wait failed. Checked on the CPU: librbgpu's host code over
emulation/host_runtime.cpp, which queues copies until they are waited for."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

CHILD = """
import ctypes, sys
sys.modules["torch"] = None  # (brings the real runtime along)
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
n, event, stream = (int(a) for a in sys.argv[2:])
import numpy as np
from robast_amd import configs
from robast_amd._lib import Context, RbError, make_rays
ctx = Context(0)
mgr = configs.c1_scene()
scene = ctx.upload(mgr.flat())
soa = {f: np.arange(n, dtype=np.float64) for f in ("x", "y", "z", "t", "dx", "dy", "dz", "lambda_")}
soa.update({f: np.arange(n, dtype=np.int32) for f in ("status", "npoints", "last_node")})
want = {f: a.copy() for f, a in soa.items()}
for ev, st in ((event, stream), (0, 0)):
    fake.fake_fail(ev, st)
    try:
        ctx.trace(scene, make_rays(soa), n, mgr.trace_opts(order=1))
        print("ok", fake.fake_pending(), fake.fake_stream_waits(), fake.fake_mallocs())
    except RbError:
        print("failed", fake.fake_pending(), fake.fake_stream_waits(), fake.fake_mallocs())
assert all((soa[f] == want[f]).all() for f in soa)
"""


@pytest.fixture(scope="module")
def host_runtime(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    so = str(tmp_path_factory.mktemp("fake") / "host_runtime.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", so,
                           os.path.join(HERE, "emulation", "host_runtime.cpp")])
    return so


def _run(so, *args):
    r = subprocess.run([sys.executable, "-c", CHILD, so] + [str(a) for a in args], capture_output=True, text=True,
                       cwd=os.path.dirname(HERE), timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    return [line.split() for line in r.stdout.splitlines()]


# 149,952 rays are 10.9 MiB of ray arrays: staged, handed back in three parts
# (an event each but the last); 250,000 are 18.1 MiB: copied array by array
@pytest.mark.parametrize("n, event, stream", [(149952, 1, 0), (149952, 2, 0), (149952, 0, 1), (149952, 0, 2),
                                              (250000, 0, 1)])
def test_no_copy_outlives_a_failed_call(host_runtime, n, event, stream):
    first, second = _run(host_runtime, n, event, stream)
    assert first[0] == "failed" and first[1] == "0"
    assert second[0] == "ok" and second[1] == "0"


@pytest.mark.parametrize("n, waits", [(1, 2), (149952, 2), (250000, 1)])
def test_a_call_waits_no_more_than_it_has_to(host_runtime, n, waits):
    """Staged: for the last part and for the timing events; array by array: once."""
    for state, pending, waited, _ in _run(host_runtime, n, 0, 0):
        assert (state, pending, int(waited)) == ("ok", "0", waits)


# ray arrays of whole and of broken steps of the work area's 256 bytes, staged
# or not
@pytest.mark.parametrize("n", [1, 64, 1000, 149952, 150001, 250001])
def test_a_second_call_allocates_nothing(host_runtime, n):
    first, second = _run(host_runtime, n, 0, 0)
    assert first[3] == "1" and second[3] == "0"
