"""The full radix sort at the edges of its two tile sizes (2048 keys up to
128 tiles, 4096 beyond), sorted and shuffled input: the order is the stable
sort of the slots by block key, an integer result compared exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,res,n", [(2, 24, 1), (2, 24, 2048), (2, 128, 2049), (3, 64, 4097),
                                       (3, 64, 128 * 2048), (3, 64, 128 * 2048 + 1)])
@pytest.mark.parametrize("shuffle", [False, True])
def test_first_order_is_the_stable_sort(dim, res, n, shuffle):
    from taichi_elements_amd import MPMSolver, mpm_solver
    mpm_solver.PRINT_PROGRESS = False
    rng = np.random.default_rng(n + shuffle)
    x = rng.uniform(0.25, 0.75, (n, dim)).astype(np.float32)
    s = MPMSolver(res=(res, ) * dim, reorder_interval=-1)
    blk = np.floor(x * np.float32(res) - np.float32(0.5)).astype(np.int64) >> 2
    if not shuffle:
        x = x[np.lexsort(blk.T)]
    s.read_restart(n, x, np.zeros_like(x), np.ones(n, np.int32), np.zeros(n, np.int32))
    s.substep(s.default_dt)
    keys, perm, orig = s.read_binning()
    blk = np.floor(x[orig] * np.float32(res) - np.float32(0.5)).astype(np.int64) >> 2
    want = np.lexsort(blk.T)
    assert np.array_equal(perm, want)
    assert np.all(np.diff(keys) >= 0)
