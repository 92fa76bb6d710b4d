"""An unbounded call that stops half way, because its particles spread over more
blocks than a window holds: the grid it leaves is that of its last substep,
bitwise the grid of a call of just those substeps."""
import ctypes

import numpy as np
import pytest

from tests.helpers import cube_particles

pytestmark = pytest.mark.gpu

DONE = 8  # substeps between two looks at the particles' box


@pytest.mark.parametrize("graphs", [False, True])
def test_grid_after_a_stopped_call(graphs):
    from taichi_elements_amd import MPMSolver, _lib, mpm_solver
    mpm_solver.PRINT_PROGRESS = False
    L = _lib.lib()
    rng = np.random.default_rng(2)
    n = 3000
    x = cube_particles(rng, n, [0.3] * 3, [0.3] * 3, 3)
    v = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
    m = rng.integers(0, 2, n).astype(np.int32)
    x[0] = 0.9
    m[0] = 1
    grids = []
    for steps in (DONE, 3 * DONE):
        s = MPMSolver(res=(32, ) * 3, unbounded=True)
        s.set_graphs(graphs)
        # one particle leaves by 300 blocks an axis in a substep
        v[0] = 300 * 4 * s.dx / s.default_dt
        s.read_restart(n, x, v, m, np.zeros(n, np.int32))
        dt = ctypes.c_float(s.default_dt)
        slow = v.copy()
        slow[0] = 0
        s.set_state(v=slow)
        assert L.mpm_substeps(s._handle, 5, dt, 0.0) == 0  # a grid of an earlier call
        assert L.mpm_sync(s._handle) == 0
        s.set_state(v=v)
        rc = L.mpm_substeps(s._handle, steps, dt, 0.0)
        assert (rc == 0) == (steps == DONE)
        assert L.mpm_sync(s._handle) != 0  # it moved more than a block
        vmax = ctypes.c_float()
        assert L.mpm_max_grid_velocity(s._handle, ctypes.byref(vmax)) == 0
        grids.append([*s.read_grid([-8] * 3, [60] * 3), np.float32(vmax.value)])
    assert grids[0][0].max() > 0
    for a, b in zip(*grids):
        assert np.array_equal(a, b)
