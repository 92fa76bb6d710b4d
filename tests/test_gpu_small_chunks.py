"""Chunks of very few particles: the solver takes any chunk >= 1, and the order
and the results do not depend on which kernel scans the block window (inside
p2g for small 2D windows, else a kernel of its own).  The order is compared
exactly with the stable sort of the previous one, the state bitwise with a twin
whose particles move every substep, which takes the scan kernel."""
import numpy as np
import pytest

from tests.helpers import cube_particles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("chunk", [1, 2, 3, 5])
def test_order_and_results(oracle, dim, chunk):
    from taichi_elements_amd import MPMSolver, mpm_solver
    mpm_solver.PRINT_PROGRESS = False
    rng = np.random.default_rng(chunk)
    n = 900
    x = cube_particles(rng, n, [0.2] * dim, [0.5] * dim, dim)
    v = (3 * rng.uniform(-1, 1, (n, dim))).astype(np.float32)
    m = rng.integers(0, 4, n).astype(np.int32)
    a, b = (MPMSolver(res=(32, ) * dim, reorder_interval=k, chunk=chunk) for k in (-1, 1))
    for s in (a, b):
        s.read_restart(n, x, v, m, np.zeros(n, np.int32))
    blo, bn = a.block_window()
    prev = None
    for step in range(4):
        x_now = a.get_state()["x"]
        for s in (a, b):
            s._run_substeps(1, a.default_dt)
        _, perm, orig = a.read_binning()
        key = oracle.block_keys(x_now, np.float32(a.inv_dx), 4, np.array(blo), np.array(bn))[orig]
        before = np.arange(n) if prev is None else prev
        np.testing.assert_array_equal(perm, before[np.argsort(key[before], kind="stable")])
        prev = perm
        sa, sb = a.get_state(), b.get_state()
        assert np.all(np.any(sa["x"] != x_now, axis=1))  # every particle moves
        for f in sa:
            assert np.array_equal(sa[f], sb[f]), (step, f)
        assert a.last_counts()["chunks"] >= n // chunk
