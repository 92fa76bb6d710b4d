"""Which way the binning goes follows the scene's last known number of chunks,
learnt by whatever call waits for the substeps: a scene of many chunks walks the
direction lists in a kernel of its own (k_members) and runs the grid operator in
a kernel, one of few chunks does both inside the transfers."""
import ctypes

import numpy as np
import pytest

from tests.helpers import cube_particles

pytestmark = pytest.mark.gpu

MANY = 2560


def _run(s, steps):
    from taichi_elements_amd import _lib
    assert _lib.lib().mpm_substeps(s._handle, steps, ctypes.c_float(s.default_dt), 0.0) == 0


def _timed(s):
    from taichi_elements_amd import _lib
    assert _lib.lib().mpm_set_timing(s._handle, 1) == 0


def _launches(s):
    names, counts, _ = s.kernel_times()
    return dict(zip(names, counts))


def _scene(chunk):
    from taichi_elements_amd import MPMSolver, mpm_solver
    mpm_solver.PRINT_PROGRESS = False
    rng = np.random.default_rng(0)
    n = 60_000
    s = MPMSolver(res=(48, ) * 3, chunk=chunk)
    s.read_restart(n, cube_particles(rng, n, [0.1] * 3, [0.8] * 3, 3),
                   np.zeros((n, 3), np.float32), np.zeros(n, np.int32), np.zeros(n, np.int32))
    return s


@pytest.mark.parametrize("wait", ["mpm_sync", "particle_info", "get_state", "last_counts"])
def test_many_chunks_are_noticed(wait):
    from taichi_elements_amd import _lib
    s = _scene(16)
    _timed(s)
    # nothing known yet: inside, but for the one that moves the particles (whose
    # order k_members finds) and the last one's grid
    _run(s, 4)
    assert _lib.lib().mpm_sync(s._handle) == 0 if wait == "mpm_sync" else getattr(s, wait)()
    _run(s, 3)
    got = _launches(s)
    assert got["k_members"] == 4 and got["k_grid_op"] == 4
    assert s.last_counts()["chunks"] > MANY
    # a new chunk size starts over
    s.set_tuning(chunk=256)
    _timed(s)
    _run(s, 4)
    got = _launches(s)
    assert "k_members" not in got and got["k_grid_op"] == 1
    assert s.last_counts()["chunks"] <= MANY


def test_few_chunks_stay_inside():
    s = _scene(256)
    s._run_substeps(4, s.default_dt)
    _timed(s)
    _run(s, 3)
    got = _launches(s)
    assert "k_members" not in got and got["k_grid_op"] == 1
