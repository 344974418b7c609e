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
                       stderr=subprocess.STDOUT, text=True, timeout=300,
                       env=dict(os.environ, PANNDE_RSG_LIB=lib, **env))
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


def test_refused_launch_is_made_by_the_per_step_kernels(lib):
    """Whatever reads or follows a launch that decided against its steps gets those steps, and those of
    the launches that were queued behind it, each with its own amplitudes and trace row."""
    run(lib, r'''
case = cases.al_block(seed=1, nx=20, ny=19, nz=18, nsteps=400, n_sensors=4)
sig = case.force[0]
def amplitude(k):
    t = 0.0
    for _ in range(k):
        t += case.dt
    return 0.125 * rsg.signal_eval(sig.signal_t, sig.signal_v, [t])[0]
row = 8 * 3 * 4
def check(n, first, base):
    assert knob("fault_velocity").value == n and knob("fault_stress").value == n
    amps = (ctypes.c_double * 4096).in_dll(rsg.lib(), "fault_amp")
    samps = (ctypes.c_double * 4096).in_dll(rsg.lib(), "fault_stress_amp")
    rows = (ctypes.c_size_t * 4096).in_dll(rsg.lib(), "fault_trace")
    for k in range(n):
        assert amps[k] == samps[k] == amplitude(first + k), k
        assert rows[k] - rows[0] == row * k
def reset(refuse, late):
    for name, v in (("refuse", refuse), ("late", late), ("resident", 0), ("velocity", 0), ("stress", 0)):
        knob("fault_" + name).value = v
reads = dict(state=lambda s: s.get_state(), traces=lambda s: s.traces(), energy=lambda s: s.energy(),
             sync=lambda s: s.synchronize(), step=lambda s: s.solve(1), zero=lambda s: s.solve(0),
             set_state=lambda s: s.set_state(np.zeros((3, case.n_nodes)), None),
             sources=lambda s: s.set_sources(case.force, []), sensors=lambda s: s.set_sensors(case.sensors))
for name, read in reads.items():
    for late in (0, 20):
        s = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64)
        reset(0, 0)
        s.solve(7)  # made
        reset(1, late)
        s.solve(9)  # not made
        assert knob("fault_resident").value == 1 and knob("fault_velocity").value == 0
        more = late and name != "zero"
        if more:  # refused behind it
            s.solve(6)
            assert knob("fault_resident").value == 2 and knob("fault_velocity").value == 0
        read(s)
        if name != "zero":  # (which may leave the decision for later)
            assert knob("fault_undecided").value == 0
            check(9 + (6 if more else 0) + (name == "step"), 7, 0)
        s.close()
# a batch takes the handle with its steps queued
s = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64)
reset(1, 20)
s.solve(9)
b = rsg.Batch(rsg.RSG_FP64)
b.remove(b.add(s, 0))
check(9, 0, 0)
b.close()
s.close()
# blocks of 256 steps: the second one is not launched resident once the first has refused
s = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64)
reset(99, 0)
s.solve(400)
assert knob("fault_resident").value == 1
check(400, 0, 0)
assert s.traces().shape[0] == 400
s.close()
# decisions that come late: blocks are queued behind the refused one, as long as its amplitudes are kept
case = cases.al_block(seed=1, nx=20, ny=19, nz=18, nsteps=1100, n_sensors=4)
s = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64)
reset(0, 0)
s.solve(20)
reset(1, 50)
s.solve(1000)
# (236 steps are left of the first amplitudes; the third upload overwrites those)
assert knob("fault_resident").value == 2
check(1000, 20, 0)
assert s.traces().shape[0] == 1020
s.close()
# many launches in one block of amplitudes: the first ones made, the rest not
s = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64)
reset(0, 0)
for _ in range(10):
    s.solve(5)
reset(1, 2000)
for _ in range(30):
    s.solve(5)
assert knob("fault_resident").value == 30 and knob("fault_velocity").value == 0
s.energy()
check(150, 50, 0)
s.close()
''')


def test_launch_without_its_event(lib):
    """A resident launch whose event could not be recorded has been made all the same: its steps and
    their time count once."""
    run(lib, r'''
case = cases.al_block(seed=1, nx=20, ny=19, nz=18, nsteps=24, n_sensors=4)
t = 0.0
s = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64)
for n, record in ((7, 2), (8, 0), (9, 1)):  # the first call's amplitude upload records an event too
    knob("fault_record").value = record
    s.solve(n)
    assert knob("fault_record").value == 0
    for _ in range(n):
        t += case.dt
    assert s.time == t
assert knob("fault_resident").value == 3 and knob("fault_velocity").value == 0
assert same(s.get_state() + (s.traces(),), case)
s.close()
''')


def test_failed_launch(lib):
    """Steps that could not be launched resident are made by the per-step kernels."""
    run(lib, r'''
case = cases.al_block(seed=1, nx=20, ny=19, nz=18, nsteps=24, n_sensors=4)
s = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64)
knob("fault_launch").value = 1
s.solve(7)
s.solve(9)
s.synchronize()
assert knob("fault_resident").value == 0 and knob("fault_velocity").value == knob("fault_stress").value == 16
s.close()
''')


def test_lost_state_is_replaced(lib):
    """A state that a launch lost is refused until both its parts have been written again, the traces
    until the sensors are set again."""
    run(lib, r'''
case = cases.al_block(seed=1, nx=20, ny=19, nz=18, nsteps=24, n_sensors=4)
rng = np.random.default_rng(3)
V, S = rng.standard_normal((3, case.n_nodes)), rng.standard_normal((6, case.n_cells))
def refused(call):
    try:
        call()
    except rsg.RSGError as e:
        return "lost" in str(e)
    return False
s = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64)
s.solve(7)
knob("fault_lost").value = 1
s.solve(8)
s.solve(1)
assert refused(s.synchronize) and refused(s.get_state) and refused(s.energy) and refused(s.traces)
s.set_state(V, None)
assert refused(s.get_state)
s.set_state(None, S)
assert all(np.array_equal(a, b) for a, b in zip(s.get_state(), (V, S)))
s.synchronize()
s.energy()
assert refused(s.traces)
s.set_sensors(case.sensors)
assert s.traces(0, 0).shape[0] == 0
assert knob("fault_resident").value == 2
s.solve(9)
assert knob("fault_resident").value == 2 and s.traces(0, 9).shape[0] == 9
# the write that replaces the state may be the first call after the loss
r = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64)
knob("fault_lost").value = 1
r.solve(8)
r.set_state(V, S)
assert all(np.array_equal(a, b) for a, b in zip(r.get_state(), (V, S)))
r.close()
s.close()
''')


def test_refused_launch_is_tried_again(lib):
    """A refused launch keeps a handle off the resident kernel for a second, not for good."""
    run(lib, r'''
import time
case = cases.al_block(seed=1, nx=20, ny=19, nz=18, nsteps=24, n_sensors=4)
s = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64)
knob("fault_refuse").value = 1
t = time.monotonic()
s.solve(7)
s.solve(7)
s.synchronize()
if time.monotonic() - t < 0.9:
    assert knob("fault_resident").value == 1 and knob("fault_velocity").value == 14
time.sleep(1.1)
n = knob("fault_velocity").value
s.solve(7)
s.synchronize()
assert knob("fault_resident").value >= 2 and knob("fault_velocity").value == n
s.close()
''')


def test_memory_of_resident_stepping(lib):
    """Set-up allocates the plan alone; the exchange buffers and the classes come with the first resident
    launch.  Where there is no memory for any of them, the per-step kernels make the steps."""
    run(lib, r'''
import time
case = cases.water_column_block(seed=9, nx=23, ny=14, nz=17, nsteps=12)
allocs, held = knob("fault_allocs"), []
for tuning in (None, dict(block_velocity=256)):  # (a named workgroup size: no plan)
    n = allocs.value
    s = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64, tuning=tuning)
    for _ in range(3):
        s.solve(1)
    held.append((allocs.value - n, s.device_bytes()))
    s.close()
assert knob("fault_velocity").value == 6 and knob("fault_resident").value == 0
# the plan: 16 bytes a cell and a tile's node, 8 a halo cell; and room for the classes' sums beside the
# amplitudes, 2 x 256 doubles each
assert held[0][0] == held[1][0] + 1 and 0 <= held[0][1] - held[1][1] <= 200 * case.n_cells + 2 * 256 * 8 * 256, held
s = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64)
n, b = allocs.value, s.device_bytes()
s.solve(case.nsteps)
assert knob("fault_resident").value == 1 and allocs.value - n == 2 and s.device_bytes() > b
assert same(s.get_state() + (s.traces(),), case)
s.close()
case.sensors = case.sensors[:0]  # (no trace buffer: nothing else is as large as the plan)
for what in ("plan", "exchange", "classes"):
    knob("fault_no_memory").value = 50 * case.n_cells if what == "plan" else 0
    s = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64)
    if what == "classes":
        s.solve(7)
        s.set_sources([], case.moment[:1])
    v, r = knob("fault_velocity").value, knob("fault_resident").value
    knob("fault_no_memory").value = knob("fault_no_memory").value or 1
    s.solve(9)
    s.synchronize()
    knob("fault_no_memory").value = 0
    assert knob("fault_velocity").value - v == 9 and knob("fault_resident").value == r
    if what == "plan":
        time.sleep(1.1)
        s.solve(9)
        s.synchronize()
        assert knob("fault_resident").value == r + 1
    s.close()
''')


def test_calls_with_another_device_current(lib):
    """Steps and state transfers use the handle's device, whichever is current, and leave that one
    current: with one transfer thread and with several."""
    run(lib, r'''
for dims in ((20, 19, 18), (46, 40, 40)):
    case = cases.al_block(seed=1, nx=dims[0], ny=dims[1], nz=dims[2], nsteps=16, n_sensors=4)
    s = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64)
    for device in (1, 0):
        rsg.lib().fault_set_device(device)
        s.set_state(np.zeros((3, case.n_nodes)), np.zeros((6, case.n_cells)))
        s.solve(8)
        now = ctypes.c_int(-1)
        state = s.get_state()
        rsg.lib().fault_get_device(ctypes.byref(now))
        assert now.value == device
        s.synchronize()
    assert knob("fault_velocity").value == 0
    s.close()
''')


def test_state_calls_wait_for_the_stream(lib):
    """rsg_get_state and rsg_set_state return with the handle's queued steps finished, also when no
    array is asked for."""
    run(lib, r'''
case = cases.al_block(seed=1, nx=9, ny=8, nz=7, nsteps=9, n_sensors=4)
s = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64)
for call in (rsg.lib().rsg_get_state, rsg.lib().rsg_set_state):
    s.solve(9)
    n = knob("fault_waits").value
    assert call(s._h, None, None) == rsg.RSG_OK
    assert knob("fault_waits").value > n
s.close()
''')


def test_transfers_share_pinned_memory(lib):
    """State transfers take their pinned chunks from a pool of the process: destroying a handle frees
    none (which would wait for every stream of the device), many handles make no more than the pool
    holds, and transfers of several threads at once move the right values."""
    run(lib, r'''
import threading
case = cases.al_block(seed=1, nx=46, ny=40, nz=40, nsteps=1, n_sensors=0)
solvers = [rsg.DeviceSolver.from_case(case, p) for p in (rsg.RSG_FP64, rsg.RSG_FP32) * 4]
bad = []
def work(i):
    rng = np.random.default_rng(i)
    for _ in range(3):
        V, S = (rng.integers(-99, 99, (k, n)).astype(float) for k, n in ((3, case.n_nodes), (6, case.n_cells)))
        solvers[i].set_state(V, S)
        if not all(np.array_equal(a, b) for a, b in zip(solvers[i].get_state(), (V, S))):
            bad.append(i)
threads = [threading.Thread(target=work, args=(i,)) for i in range(len(solvers))]
for t in threads:
    t.start()
for t in threads:
    t.join()
assert not bad and 1 <= knob("fault_pinned").value <= 16
for s in solvers:
    s.close()
assert knob("fault_unpinned").value == 0
''')


def test_status_words_are_shared(lib):
    """Handles that step resident take their status words from pages of the process: destroying one
    frees no pinned memory, and the words serve the next handle, zeroed."""
    run(lib, r'''
case = cases.al_block(seed=1, nx=9, ny=8, nz=7, nsteps=9, n_sensors=4)
case.force = []  # no sources: no pinned staging of amplitudes either
def stepped():
    s = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64)
    s.solve(9)
    s.synchronize()
    return s
solvers = [stepped() for _ in range(100)]
assert knob("fault_resident").value == 100 and knob("fault_pinned").value == 2
knob("fault_lost").value = 1
lost = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64)
lost.solve(9)
for s in solvers + [lost]:
    s.close()
solvers = [stepped() for _ in range(128)]
assert knob("fault_pinned").value == 2
for s in solvers:
    s.close()
assert knob("fault_unpinned").value == 0
''')


def test_state_without_memory_for_the_transfer(lib):
    """A state can be read and written when the device is full or no memory can be pinned, and goes
    through the device again once there is some."""
    run(lib, r'''
rng = np.random.default_rng(3)
for precision in (rsg.RSG_FP64, rsg.RSG_FP32):
    for lack in ("fault_no_memory", "fault_no_pinned"):
        case = cases.al_block(seed=1, nx=46, ny=40, nz=40, nsteps=1, n_sensors=0)
        s = rsg.DeviceSolver.from_case(case, precision)
        for n in (1, 0, 0):
            knob(lack).value = n
            V, S = (rng.integers(-99, 99, (k, n)).astype(float) for k, n in ((3, case.n_nodes), (6, case.n_cells)))
            s.set_state(V, S)
            assert all(np.array_equal(a, b) for a, b in zip(s.get_state(), (V, S))), lack
        s.close()
assert knob("fault_pinned").value > 0
''')
