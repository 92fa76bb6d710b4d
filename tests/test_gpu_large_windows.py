"""The block scan at the edges of its ranges: windows of the most blocks that one
pass takes, one tile more, groups of tiles that are full, one over and partly
empty, and millions of blocks, with particles all over the window.  The order is
compared exactly with a stable sort, the counts with numpy's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TILE, ONE_PASS, GROUP = 512, 448, 128  # blocks a tile, tiles in one pass, tiles a group


@pytest.mark.parametrize("res", [
    (1772, 2028),   # 448 tiles
    (1776, 2028),   # 449
    (2028, 2028),   # 512, four full groups
    (2032, 2028),   # 513
    (15980, 3980),  # 7813
    (40, 13000, 8),
])
def test_order_and_counts(oracle, res):
    from taichi_elements_amd import MPMSolver, mpm_solver
    mpm_solver.PRINT_PROGRESS = False
    d = len(res)
    blocks = int(np.prod([(r + 3) // 4 + 5 for r in res]))
    print("tiles", -(-blocks // TILE), flush=True)
    rng = np.random.default_rng(blocks)
    n = 30_000
    s = MPMSolver(res=res, reorder_interval=-1)
    size = np.asarray(res) * s.dx
    x = (rng.uniform(0.02, 0.98, (n, d)) * size).astype(np.float32)
    x[:4] = (np.full(d, 5 * s.dx), size - 5 * s.dx, 0.5 * size, 0.3 * size)
    x[n // 2:] = (0.5 * size + rng.uniform(-20, 20, (n - n // 2, d)).clip(-3, 3) * s.dx)
    v = (0.5 * s.dx / s.default_dt * rng.uniform(-1, 1, (n, d))).astype(np.float32)
    s.read_restart(n, x, v, np.zeros(n, np.int32), np.zeros(n, np.int32))
    blo, bn = s.block_window()
    assert int(np.prod(bn)) == blocks
    prev = None
    for _ in range(3):
        x_now = s.get_state()["x"]
        s._run_substeps(1, s.default_dt)
        keys, perm, orig = s.read_binning()
        key = oracle.block_keys(x_now, np.float32(s.inv_dx), 4, np.array(blo), np.array(bn))[orig]
        before = np.arange(n) if prev is None else prev
        np.testing.assert_array_equal(perm, before[np.argsort(key[before], kind="stable")])
        np.testing.assert_array_equal(keys, key[perm])
        prev = perm
        used, count = np.unique(key, return_counts=True)
        stride = np.concatenate([[1], np.cumprod(bn[:d])[:-1]])
        reach = {int(b + np.dot(o, stride)) for o in np.ndindex(*(2, ) * d) for b in used}
        chunk = s.tuning()[0]
        assert s.last_counts() == dict(valid=n, chunks=int((-(-count // chunk)).sum()),
                                       active_blocks=len(reach), particle_blocks=len(used))
