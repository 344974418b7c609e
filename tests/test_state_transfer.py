"""States written and read back through the device's reordering (rsg_state.hip): every value in
its place, in one chunk and in several, each array alone, for both precisions."""
import ctypes

import numpy as np
import pytest

from pannde_amd import cases, rsg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [rsg.RSG_FP64, rsg.RSG_FP32])
@pytest.mark.parametrize("dims", [(1, 1, 1), (9, 7, 5), (37, 31, 29), (70, 60, 61)])
def test_round_trip(dims, precision):
    """1 cell to 2.3 M values: a chunk holds 256 Ki, a second thread starts at 256 Ki."""
    case = cases.al_block(seed=1, nx=dims[0], ny=dims[1], nz=dims[2], nsteps=1, n_sensors=1)
    s = rsg.DeviceSolver.from_case(case, precision)
    rng = np.random.default_rng(3)
    V = rng.standard_normal((3, case.n_nodes))
    S = 1e6 * rng.standard_normal((6, case.n_cells))
    V[:, 0] = np.inf, -0.0, np.nan
    S[5, -1] = -np.inf
    if precision == rsg.RSG_FP32:
        V, S = V.astype(np.float32).astype(np.float64), S.astype(np.float32).astype(np.float64)
    s.set_state(V, S)
    for _ in range(2):
        V1, S1 = s.get_state()
        assert V1.tobytes() == V.tobytes() and S1.tobytes() == S.tobytes()
    s.set_state(2 * V, None)
    s.set_state(None, -S)
    only = np.empty_like(S)
    assert rsg.lib().rsg_get_state(s._h, None, only.ctypes.data_as(ctypes.POINTER(ctypes.c_double))) == rsg.RSG_OK
    V1, S1 = s.get_state()
    assert np.array_equal(V1, 2 * V, equal_nan=True) and np.array_equal(S1, -S) and np.array_equal(only, -S)
    s.close()
