"""Per-cell stiffness arrays that hold the nine axial entries alone, and all 21."""
import numpy as np
import pytest

from oracle import oracle_rsg as orc
from pannde_amd import cases, rsg


def graded(kind):
    """A block no two cells of which share a stiffness; C16 zero, one value or varying too."""
    case = cases.al_block(seed=4, nx=17, ny=9, nz=8, nsteps=15, n_sensors=5)
    nc = case.cells.shape[0]
    scale = 1 - 0.3 * np.random.default_rng(1).random(nc)
    case.cij = [cases.Field(cases.FIELD_CELL, np.broadcast_to(f.data, nc) * scale) for f in case.cij]
    c16 = cases.CIJ_PAIRS.index((0, 5))
    if kind != "axial":
        case.cij[c16] = cases.Field(cases.FIELD_CELL, 2.0e9 * (np.ones(nc) if kind == "constant" else scale))
    return case


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [rsg.RSG_FP64, rsg.RSG_FP32])
@pytest.mark.parametrize("kind", ["axial", "constant", "varying"])
def test_per_cell_stiffness(kind, precision):
    """Per-step kernels staged and not, both layouts of C, the resident kernel and a batch: FP64 as the
    oracle bit for bit, FP32 alike among themselves; energies alike."""
    case = graded(kind)
    V, S, _, traces = orc.run_oracle(case)
    out = []
    for tuning in (dict(block_velocity=256), dict(block_velocity=256, c_layout=-1),
                   dict(lds_velocity=-1, lds_stress=-1), dict(per_thread_stress=2), None):
        s = rsg.DeviceSolver.from_case(case, precision, tuning=tuning)
        s.solve(case.nsteps)
        out.append(s.get_state() + (s.traces(), np.array(s.energy())))
        s.close()
    b = rsg.Batch(precision)
    slot = b.add(rsg.DeviceSolver.from_case(case, precision), case.nsteps)
    b.run(10)
    b.synchronize()
    s = b.remove(slot)
    out.append(s.get_state() + (s.traces(), np.array(s.energy())))
    b.close()
    s.close()
    ref = (V, S, traces) if precision == rsg.RSG_FP64 else out[0][:3]
    for i, o in enumerate(out):
        assert all(np.array_equal(x, y) for x, y in zip(o[:3], ref)), i
        assert np.array_equal(o[3], out[0][3]) and np.isfinite(o[3]).all(), i
