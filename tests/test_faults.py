"""What the host code does when the system refuses it something: on the CPU, over the stand-ins for
the HIP runtime (tests/sanitize/hip_host_stub.cpp, resident_stub.cpp), with failures on demand
(tests/sanitize/faults.cpp).  Each script runs in a process of its own."""
import os
import re
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "pannde_amd", "csrc")
HERE = os.path.join(ROOT, "tests", "sanitize")

pytestmark = [pytest.mark.timeout(600),
              pytest.mark.skipif(shutil.which("g++") is None or
                                 not os.path.exists("/opt/rocm/include/hip/hip_runtime_api.h"),
                                 reason="needs g++ and the HIP headers")]


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("faults") / "libfaults.so")
    with open(os.path.join(HERE, "faults.cpp")) as f:
        text = f.read()
    wrapped = set(re.findall(r"__wrap_(\w+)\(", text)) | set(re.findall(r"#define [A-Z_0-9]+ (_Z\w+)", text))
    cmd = ["g++", "-x", "c++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__",
           "-I/opt/rocm/include", os.path.join(CSRC, "rsg_host.cpp"), os.path.join(HERE, "hip_host_stub.cpp"),
           os.path.join(HERE, "resident_stub.cpp"), os.path.join(HERE, "faults.cpp"), "-o", out, "-lpthread"]
    r = subprocess.run(cmd + ["-Wl,--wrap=" + w for w in sorted(wrapped)], stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-4000:]
    return out


PRELUDE = r'''
import ctypes, sys
import numpy as np
sys.path[:0] = [sys.argv[1], sys.argv[1] + "/tests"]
from oracle import oracle_rsg as orc
from pannde_amd import cases, rsg
def knob(name):
    return ctypes.c_int.in_dll(rsg.lib(), name)
def same(got, case):
    V0, S0, t0, tr0 = orc.run_oracle(case)
    return np.array_equal(got[0], V0) and np.array_equal(got[1], S0) and np.array_equal(got[2], tr0)
'''


def run(lib, script, **env):
    r = subprocess.run([sys.executable, "-c", PRELUDE + script + '\nprint("ok")\n', ROOT], stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=300, env=dict(os.environ, PANNDE_RSG_LIB=lib, **env))
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout[-4000:]


def test_set_up_without_threads(lib):
    """No thread, or only some, to be had: the set-up makes all its parts on those it has."""
    run(lib, r'''
case = cases.al_block(seed=1, nx=30, ny=28, nz=26, nsteps=9, n_sensors=4)
for n in (0, 1, 2, 3, 5):
    knob("fault_threads").value = n
    s = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64)
    s.solve(case.nsteps)
    assert same(s.get_state() + (s.traces(),), case), n
    s.close()
''')
