"""mpm_read_max_velocity at the edges of its count: none (zero or less: it waits
and reports errors), one, all of a long call (more entries than the pinned words
a handle starts with) and more than were run, through the C ABI."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_counts():
    from taichi_elements_amd import MPMSolver, _lib, mpm_solver
    mpm_solver.PRINT_PROGRESS = False
    L = _lib.lib()
    rng = np.random.default_rng(0)
    n = 2000
    s = MPMSolver(res=(32, 32))
    x = rng.uniform(0.3, 0.7, (n, 2)).astype(np.float32)
    s.read_restart(n, x, np.full((n, 2), 0.5, np.float32), np.zeros(n, np.int32),
                   np.zeros(n, np.int32))
    assert L.mpm_read_max_velocity(s._handle, 0, None) == 0
    assert L.mpm_read_max_velocity(s._handle, 1, _lib.fptr(np.zeros(1, np.float32))) != 0
    steps = 300
    assert L.mpm_substeps(s._handle, steps, ctypes.c_float(s.default_dt), 0.0) == 0
    for k in (0, -1, -2, -1000):
        assert L.mpm_read_max_velocity(s._handle, k, None) == 0
    out = np.full(steps + 1, np.nan, np.float32)
    assert L.mpm_read_max_velocity(s._handle, steps, _lib.fptr(out)) == 0
    assert np.all(out[:steps] > 0) and np.isnan(out[steps])
    one = np.zeros(1, np.float32)
    assert L.mpm_read_max_velocity(s._handle, 1, _lib.fptr(one)) == 0
    assert one[0] == out[0]
    assert np.abs(s.get_state()["v"]).max() == out[steps - 1]
    assert L.mpm_read_max_velocity(s._handle, steps + 1, _lib.fptr(out)) != 0
    assert L.mpm_read_max_velocity(s._handle, 1, None) != 0
