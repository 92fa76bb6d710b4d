"""The steady-state binning (the previous substep's direction lists) against
numpy's stable sort by block key, at the edges of its dispatch: particle
counts on both sides of the line between the lists walked inside the
transfer and by a kernel of their own, chunks of 16 particles in dense blocks
(more than 64 groups per block, so several rounds), chunks of several
batches, and substeps that move the particles."""
import numpy as np
import pytest

from tests.helpers import cube_particles

pytestmark = pytest.mark.gpu

# particles up to which the transfer walks the lists (use_g2p2g, p2g)
LINE, P2G_LINE = 160 * 1024, 256 * 1024


@pytest.fixture(autouse=True)
def _quiet():
    from taichi_elements_amd import mpm_solver
    mpm_solver.PRINT_PROGRESS = False


CASES = [
    # dim, res, n, side, chunk, reorder_interval, options
    (2, 48, 1, 0.2, 256, -1, {}),
    (2, 48, 3001, 0.15, 16, -1, {}),
    (2, 64, 40000, 0.3, 1024, 3, {}),
    (3, 24, 20011, 0.3, 16, -1, {}),
    (3, 24, 20011, 0.3, 16, 2, {}),
    (3, 32, 60000, 0.25, 1024, -1, {}),
    (3, 48, LINE, 0.4, 256, -1, {}),
    (3, 48, LINE + 1, 0.4, 256, -1, {}),
    (3, 48, LINE + 1, 0.2, 1000, 2, {}),
    (3, 48, P2G_LINE, 0.5, 256, -1, {}),
    (3, 48, P2G_LINE + 1, 0.5, 256, -1, {}),
    (3, 48, 60000, 0.6, 16, -1, {}),  # more chunks than the transfer walks the lists for
    (3, 32, 9001, 0.3, 64, 2, dict(use_g2p2g=True)),
    (3, 48, LINE + 1, 0.4, 256, -1, dict(use_g2p2g=True)),
    (3, 32, 9001, 0.3, 64, 2, dict(quant=True)),
]


@pytest.mark.parametrize("dim,res,n,side,chunk,interval,options", CASES)
def test_order_is_stable_sort_of_previous_order(oracle, dim, res, n, side, chunk, interval,
                                                options):
    from taichi_elements_amd import MPMSolver
    rng = np.random.default_rng(n)
    s = MPMSolver(res=(res, ) * dim, reorder_interval=interval, chunk=chunk, **options)
    x = cube_particles(rng, n, [0.5 - side / 2] * dim, [side] * dim, dim)
    v = (3 * rng.uniform(-1, 1, (n, dim))).astype(np.float32)
    s.read_restart(n, x, v, np.zeros(n, np.int32), np.zeros(n, np.int32))
    blo, bn = s.block_window()
    perm_prev = orig_prev = None
    for step in range(7):
        x_now = s.get_state()["x"]
        s.substep(s.default_dt)
        keys, perm, orig = s.read_binning()
        key_slot = oracle.block_keys(x_now, np.float32(s.inv_dx), 4, np.array(blo),
                                     np.array(bn))[orig]
        if step == 0:
            prev = np.arange(n)
        else:
            # the previous order, as slots of this substep
            slot = np.empty(n, np.int64)
            slot[orig] = np.arange(n)
            prev = slot[orig_prev[perm_prev]]
        expected = prev[np.argsort(key_slot[prev], kind="stable")]
        np.testing.assert_array_equal(perm, expected)
        np.testing.assert_array_equal(keys, key_slot[perm])
        perm_prev, orig_prev = perm, orig
    if interval > 0 and n > 1:  # the particles were moved into the sorted order
        assert not np.array_equal(orig, np.arange(n))
