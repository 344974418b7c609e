"""A HIP error that another call of the thread left behind is not taken for a state transfer's."""
import ctypes

import numpy as np
import pytest

from pannde_amd import cases, rsg

pytestmark = pytest.mark.gpu


def test_state_after_a_failed_allocation():
    case = cases.al_block(seed=1, nx=9, ny=7, nz=5, nsteps=1, n_sensors=1)
    s = rsg.DeviceSolver.from_case(case, rsg.RSG_FP64)
    rng = np.random.default_rng(3)
    V, S = rng.standard_normal((3, case.n_nodes)), rng.standard_normal((6, case.n_cells))
    hip, p = ctypes.CDLL("libamdhip64.so"), ctypes.c_void_p()
    for _ in range(2):
        assert hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(1 << 50)) != 0  # more than any GPU has
        s.set_state(V, S)
        V1, S1 = s.get_state()
        assert np.array_equal(V1, V) and np.array_equal(S1, S)
    hip.hipGetLastError()
    s.close()
