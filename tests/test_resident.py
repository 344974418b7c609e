"""Resident stepping (rsg_resident.hip): many steps of a mesh in one launch, its tiles in LDS.

On the CPU the set-up's plan is walked by a stand-in for the kernel (tests/sanitize/
resident_stub.cpp), tile by tile with every index checked, and the result compared bit for bit
with the oracle.  On the GPU the kernel is compared bit for bit with the per-step kernels (a
handle whose tuning names a workgroup size uses those) and with the oracle."""
import os
import shutil
import subprocess
import sys

import numpy as np
import pytest

from conftest import load_golden
from oracle import oracle_rsg as orc
from pannde_amd import cases, rsg

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def jobs(name):
    if name == "one_cell":
        return cases.al_block(seed=1, nx=1, ny=1, nz=1, nsteps=9, n_sensors=2)
    if name == "one_tile":  # 500 cells: the most that one tile takes
        return cases.al_block(seed=2, nx=10, ny=10, nz=5, nsteps=13, n_sensors=200)
    if name == "two_tiles":
        return cases.water_column_block(seed=3, nx=8, ny=9, nz=7, nsteps=11)
    if name == "flat":
        return cases.al_block(seed=4, nx=61, ny=47, nz=1, nsteps=9, n_sensors=7)
    if name == "cracked_plate":
        return cases.cfrp_plate(seed=3, nx=40, ny=36, cells_per_ply=1, nsteps=12, n_holes=2, renumber=True,
                                crack=cases.Crack((1e-3, 0.9e-3, 16 * 5e-5), 30.0, 0.8e-3, 4e-4))
    if name == "bracket":
        return cases.ti_bracket(seed=7, leg=48, width=12, height=9, nsteps=11)
    if name == "moments":
        return cases.water_column_block(seed=9, nx=23, ny=14, nz=17, nsteps=9)
    if name == "rest":  # sensors, no source
        case = cases.al_block(seed=5, nx=12, ny=11, nz=9, nsteps=8, n_sensors=5)
        case.force = []
        return case
    return load_golden(name)[0]


NAMES = ("one_cell", "one_tile", "two_tiles", "flat", "cracked_plate", "bracket", "moments", "rest",
         "water_column_nodec", "three_transducers")

SCRIPT = r'''
import sys
import numpy as np
sys.path[:0] = [sys.argv[1], sys.argv[1] + "/tests"]
import test_resident
from oracle import oracle_rsg as orc
from pannde_amd import rsg
for name in test_resident.NAMES:
    case = test_resident.jobs(name)
    V0, S0, t0, tr0 = orc.run_oracle(case)
    for tuning in (None, dict(coeff_classes=-1), dict(coeff_classes=-1, c_layout=-1)):
        s = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64, tuning=tuning)
        s.solve(case.nsteps)
        V, S = s.get_state()
        tr = s.traces()
        s.close()
        assert np.array_equal(V, V0) and np.array_equal(S, S0) and np.array_equal(tr, tr0), (name, tuning)
        f = rsg.DeviceSolver.from_case(case, rsg.RSG_FP32, tuning=tuning)
        f.solve(case.nsteps)
        # FP32 fields after a few steps: a few roundings of 2^-24 each against FP64
        err = np.abs(f.get_state()[0] - V0).max() / max(np.abs(V0).max(), 1e-300)
        assert err < 1e-5, (name, tuning, err)
        f.close()
print("ok")
'''


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.exists("/opt/rocm/include/hip/hip_runtime_api.h"),
                    reason="needs g++ and the HIP headers")
@pytest.mark.timeout(600)
def test_plan_steps_as_the_oracle(tmp_path):
    lib = str(tmp_path / "libstub.so")
    here = os.path.join(ROOT, "tests", "sanitize")
    cmd = ["g++", "-x", "c++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__",
           "-I/opt/rocm/include", os.path.join(ROOT, "pannde_amd", "csrc", "rsg_host.cpp"),
           os.path.join(here, "hip_host_stub.cpp"), os.path.join(here, "resident_stub.cpp"), "-o", lib, "-lpthread"]
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-4000:]
    # 256 compute units, and 24: larger tiles (the plate: 900 cells each)
    for cus in ("256", "24"):
        env = dict(os.environ, PANNDE_RSG_LIB=lib, RESIDENT_CUS=cus)
        r = subprocess.run([sys.executable, "-c", SCRIPT, ROOT], stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                           text=True, timeout=500, env=env)
        assert r.returncode == 0 and r.stdout.strip().endswith("ok"), (cus, r.stdout[-4000:])


def run(case, precision, tuning, chunks):
    s = rsg.DeviceSolver.from_case(case, precision, tuning=tuning)
    for n in chunks:
        s.solve(n)
    out = s.get_state() + (s.traces(), s.time)
    s.close()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [rsg.RSG_FP64, rsg.RSG_FP32])
@pytest.mark.parametrize("name", NAMES)
def test_resident_equals_per_step_kernels(name, precision):
    """Also split into calls of few and many steps, so that resident and per-step launches (and their
    amplitude windows) follow each other, and with per-entity coefficients."""
    case = jobs(name)
    case.nsteps = 40
    ref = run(case, precision, dict(block_velocity=256, block_stress=256), [40])
    if precision == rsg.RSG_FP64:
        V0, S0, t0, tr0 = orc.run_oracle(case)
        assert all(np.array_equal(a, b) for a, b in zip(ref, (V0, S0, tr0))) and ref[3] == t0
    for chunks in ([40], [7, 1, 13, 2, 17]):
        for tuning in (None, dict(coeff_classes=-1)):
            got = run(case, precision, tuning, chunks)
            assert all(np.array_equal(a, b) for a, b in zip(got, ref)), (chunks, tuning)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [rsg.RSG_FP64, rsg.RSG_FP32])
@pytest.mark.parametrize("name", ("two_tiles", "cracked_plate", "moments", "rest"))
def test_launch_that_decides_against_its_steps(name, precision, monkeypatch):
    """Tiles that do not get onto the GPU together: one workgroup makes the steps, and the handle
    goes on with the per-step kernels."""
    case = jobs(name)
    for tuning in (None, dict(coeff_classes=-1)):
        per_step = dict(block_velocity=256, block_stress=256, **(tuning or {}))
        ref = run(case, precision, per_step, [7, 9, 6])
        with monkeypatch.context() as m:
            m.setenv("PANNDE_RSG_RESIDENT", "alone")
            got = run(case, precision, tuning, [7, 9, 6])
        assert all(np.array_equal(a, b) for a, b in zip(got, ref)), tuning


@pytest.mark.gpu
def test_handles_on_several_threads():
    """Resident launches of several handles take turns on the GPU."""
    import threading

    case = jobs("moments")
    ref = run(case, rsg.RSG_FP64, dict(block_velocity=256, block_stress=256), [60])
    out = [None] * 5

    def work(i):
        out[i] = run(case, rsg.RSG_FP64, None, [20, 5, 6, 9, 20])

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(out))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(o is not None and all(np.array_equal(a, b) for a, b in zip(o, ref)) for o in out)


@pytest.mark.gpu
@pytest.mark.parametrize("precision,dims", [(rsg.RSG_FP64, (64, 52, 41)), (rsg.RSG_FP64, (80, 71, 57)),
                                            (rsg.RSG_FP32, (80, 71, 57)), (rsg.RSG_FP32, (97, 83, 66))])
def test_resident_at_its_largest(precision, dims):
    """Tiles whose records are in LDS and tiles whose are not, up to the last sizes that fit."""
    case = cases.al_block(seed=6, nx=dims[0], ny=dims[1], nz=dims[2], nsteps=300, n_sensors=9)
    ref = run(case, precision, dict(block_velocity=256, block_stress=256), [300])
    got = run(case, precision, None, [300])
    assert all(np.array_equal(a, b) for a, b in zip(got, ref))


def graded_mesh(classes, scale):
    """A block of 260 x 6 x 5 cells with `classes` spacings along x, its lengths times `scale`."""
    case = cases.al_block(seed=8, nx=260, ny=6, nz=5, nsteps=6, n_sensors=3)
    rng = np.random.default_rng(classes)
    widths = rng.choice(rng.uniform(0.6e-4, 2.0e-4, classes), 260)
    case.x = np.concatenate([[0.0], np.cumsum(widths)])[np.rint(case.x / 1e-4).astype(int)] * scale
    case.y, case.z = case.y * scale, case.z * scale
    case.force = []
    return case


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [rsg.RSG_FP64, rsg.RSG_FP32])
@pytest.mark.parametrize("classes,scale", [(1, 1.0), (5, 1.0), (40, 1.0), (260, 1.0), (5, 1e-17), (1, 2.0 ** 70)])
def test_quotients_of_any_size(classes, scale, precision):
    """Spacings from the LDS tables, the caches and per-node arrays, usual and not, and states whose
    values lie anywhere between the denormals and infinity: each difference quotient is the rounded
    quotient of the per-step kernels (and the oracle)."""
    case = graded_mesh(classes, scale)
    rng = np.random.default_rng(3)
    nn, nc = case.x.shape[0], case.cells.shape[0]
    top = 1000 if precision == rsg.RSG_FP64 else 100
    for low, special in ((-1074, False), (-1000, False), (-900, True), (0, True)):
        V, S = (rng.uniform(-2, 2, (k, n)) * 2.0 ** rng.integers(max(low, -1070), top if low == 0 else low + 200, (k, n))
                for k, n in ((3, nn), (6, nc)))
        for a in (V, S):
            a[rng.random(a.shape) < 0.3] = 0.0
            if special:
                a[rng.random(a.shape) < 1e-3] = np.inf
                a[rng.random(a.shape) < 1e-3] = np.nan
        out = []
        for tuning in (dict(block_velocity=256, block_stress=256), None):
            s = rsg.DeviceSolver.from_case(case, precision, tuning=tuning)
            s.set_state(V, S)
            s.solve(6)
            out.append(s.get_state() + (s.traces(),))
            s.close()
        assert all(np.array_equal(a, b, equal_nan=True) for a, b in zip(*out)), low
