"""The C ABI's host code over a HIP runtime in host memory (tests/host/fake_hip.cpp),
for tests that need no GPU: allocations that fail, what a call holds, which calls are
refused.  Each test body runs in a process of its own."""
import os
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "tdlbcpp_amd", "csrc")
SOURCES = ("capi", "batch", "server", "rushton", "readback")

PRELUDE = """
import ctypes, sys
sys.path.insert(0, {root!r})
import numpy as np
import tdlbcpp_amd as td
td.LIB_PATH = {lib!r}
L = td.lib()
NOMEM, STATE = -3, -4  # TDLB_ERR_NOMEM, TDLB_ERR_STATE
for _n in ("malloc", "pinned", "new"):
    getattr(L, "fake_fail_" + _n).argtypes = [ctypes.c_int64]
L.fake_limit.argtypes = [ctypes.c_uint64]
for _n in ("live", "peak"):
    getattr(L, "fake_" + _n).restype = ctypes.c_uint64
for _n in ("mallocs", "pinned", "pinned_mallocs", "gathers"):
    getattr(L, "fake_" + _n).restype = ctypes.c_int64

def tank(T, prec=td.PREC_F32, bind=True, **kw):
    cu = td.ComputeUnit(T, precision=prec, **kw)
    cu.initialise(1.0)
    if bind:
        cu.bind_rushton(td.rushton_defaults(T))
    return cu
"""


@pytest.fixture(scope="session")
def host_library(tmp_path_factory):
    """run(*bodies): the Python code of a test over the host library, in a child process"""
    out = tmp_path_factory.mktemp("host")
    flags = ["-D__HIP_PLATFORM_AMD__", "-D__align__(n)=__attribute__((aligned(n)))", "-DHIP_SYMBOL(x)=(x)",
             "-I/opt/rocm/include", "-O1", "-std=c++17", "-fPIC", "-ffp-contract=off", "-w"]
    jobs = []
    for name, src in [(s, os.path.join(CSRC, s + ".cpp")) for s in SOURCES] + \
                     [("fake_hip", os.path.join(ROOT, "tests", "host", "fake_hip.cpp"))]:
        obj = str(out / (name + ".o"))
        jobs.append((obj, subprocess.Popen(["g++"] + flags + ["-c", "-o", obj, src])))
    assert [p.wait() for _, p in jobs] == [0] * len(jobs)
    lib = str(out / "libhost.so")
    subprocess.run(["g++", "-shared", "-pthread", "-Wl,-Bsymbolic,-z,defs", "-o", lib] + [o for o, _ in jobs],
                   check=True)

    def run(*bodies, timeout=120):
        code = PRELUDE.format(root=ROOT, lib=lib) + "".join(textwrap.dedent(b) for b in bodies)
        r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=timeout)
        assert r.returncode == 0, f"exit {r.returncode}\n{r.stdout}\n{r.stderr[-4000:]}"

    return run
