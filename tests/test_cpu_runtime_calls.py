"""The host side of the single-matrix calls against a HIP runtime of host
functions (hip_host_shim.cpp): what is left after a call that fails, and what
the next call does about it.  Kernels do not run, so a call that gets as far
as waiting for one reports that its record is missing."""
import os
import shutil
import subprocess
import sys

import pytest

from conftest import PKG, ROOT

HIPCC = "/opt/rocm/bin/hipcc"
needs_hip = pytest.mark.skipif(not (shutil.which("g++") and os.path.exists(HIPCC)),
                               reason="no HIP headers or compiler")

PRELUDE = """
import ctypes, sys
import numpy as np
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
shim.shim_log.restype = ctypes.c_char_p
sys.path.insert(0, sys.argv[2])
import permanent_amd as P
def error(fn):
    try:
        fn()
    except P.PermError as e:
        return str(e)
    return None
def calls():
    log = shim.shim_log().decode().split()
    shim.shim_clear()
    return log
real = 1.0 + np.arange(64.0).reshape(8, 8) % 5
ones = np.eye(20, dtype=np.int32)
ones[:, 0] = 1
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    so = tmp_path_factory.mktemp("shim") / "libhip_host_shim.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", os.path.join(ROOT, "tests", "hip_host_shim.cpp"),
                    "-o", str(so)], check=True)
    return str(so)


def run(shim, body):
    p = subprocess.run([sys.executable, "-c", PRELUDE + body, shim, PKG], text=True,
                       capture_output=True, timeout=120)
    assert p.returncode == 0, (p.returncode, p.stdout, p.stderr[-2000:])


@needs_hip
@pytest.mark.parametrize("name,after", [("hipStreamCreateWithFlags", 0), ("hipEventCreate", 0),
                                        ("hipEventCreate", 1), ("hipHostMalloc", 0),
                                        ("hipMalloc", 0), ("hipHostMalloc", 1)])
@pytest.mark.parametrize("call", ["P.dense(real)", "P.skip(ones)"])
def test_call_after_a_failed_first_call(shim, name, after, call):
    """A first call that fails to get its stream, events, record or memory
    returns an error; the next one starts over (it did not find the record)."""
    run(shim, f"""
shim.shim_fail(b"{name}", {after})
first = error(lambda: {call})
assert first and "shim" in first, first
for again in range(2):
    e = error(lambda: {call})
    assert e and "without its record" in e, e
made = calls()
live = made.count("hipStreamCreateWithFlags") - made.count("hipStreamDestroy")
events = made.count("hipEventCreate") - made.count("hipEventDestroy")
failed = {{"hipStreamCreateWithFlags": (1, 0), "hipEventCreate": (0, 1)}}.get("{name}", (0, 0))
assert (live, events) == (1 + failed[0], 2 + failed[1]), (made, live, events)
""")


@needs_hip
def test_call_after_a_chunked_one_does_not_wait(shim):
    """A chunked run waits for its last kernel: the call after it finds the
    stream idle and starts without another wait; after one that failed midway
    it waits first."""
    run(shim, """
P.chunked(real)
calls()
error(lambda: P.dense(real))
log = calls()
assert log.index("hipLaunchKernel") < log.index("hipStreamSynchronize"), log
shim.shim_fail(b"hipEventRecord", 1)
assert error(lambda: P.chunked(real))
calls()
error(lambda: P.dense(real))
log = calls()
assert log.index("hipStreamSynchronize") < log.index("hipLaunchKernel"), log
""")
