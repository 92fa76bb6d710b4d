"""The block scan inside p2g (2D, steady state) at the edges of its range: the
smallest window and those with the most blocks it takes and one more, more
chunks than workgroups, one particle, scenes of a batch that sit a call out.
The order is compared exactly with the stable sort of the previous one; the
state and the grid are bitwise those of a twin whose particles move every
substep, which takes the scan kernel."""
import numpy as np
import pytest

from tests.helpers import cube_particles

pytestmark = pytest.mark.gpu

LINE = 256 * 1024  # particles up to which p2g walks the lists


@pytest.fixture(autouse=True)
def _quiet():
    from taichi_elements_amd import batch, mpm_solver
    mpm_solver.PRINT_PROGRESS = batch.PRINT_PROGRESS = False


@pytest.mark.parametrize("res,n,side,chunk,options", [
    ((8, 8), 1, 0.3, 256, {}),
    ((16, 16), 700, 0.6, 16, {}),
    ((62, 70), 5000, 0.5, 64, {}),
    ((128, 128), 40000, 0.8, 16, {}),           # more chunks than workgroups
    ((168, 168), 20000, 0.8, 256, {}),
    ((176, 168), 3000, 0.8, 256, dict(quant=True)),
    ((184, 184), 20000, 0.8, 256, {}),          # past the range
    ((160, 160), LINE, 0.8, 1024, {}),
    ((160, 160), LINE + 1, 0.8, 1000, {}),
    ((128, 128), LINE, 0.9, 16, {}),            # more chunks than the lists are walked for
])
def test_order_and_results(oracle, res, n, side, chunk, options):
    from taichi_elements_amd import MPMSolver
    rng = np.random.default_rng(n + chunk)
    x = cube_particles(rng, n, [0.5 - side / 2] * 2, [side] * 2, 2)
    x[:, 1] *= min(res[1] / res[0], 1.0)
    v = (3 * rng.uniform(-1, 1, (n, 2))).astype(np.float32)
    m = rng.integers(0, 5, n).astype(np.int32)
    a, b = (MPMSolver(res=res, reorder_interval=k, chunk=chunk, **options) for k in (-1, 1))
    for s in (a, b):
        s.read_restart(n, x, v, m, np.zeros(n, np.int32))
    blo, bn = a.block_window()
    print("blocks", int(np.prod(bn)), flush=True)
    prev = None
    for step in range(5):
        x_now = a.get_state()["x"]
        for s in (a, b):
            s._run_substeps(1, a.default_dt)
        keys, perm, orig = a.read_binning()
        key = oracle.block_keys(x_now, np.float32(a.inv_dx), 4, np.array(blo), np.array(bn))[orig]
        before = np.arange(n) if prev is None else prev
        np.testing.assert_array_equal(perm, before[np.argsort(key[before], kind="stable")])
        np.testing.assert_array_equal(keys, key[perm])
        prev = perm
        sa, sb = a.get_state(), b.get_state()
        for f in sa:
            assert np.array_equal(sa[f], sb[f]), (step, f)
        lo, size = [-8] * 2, [r + 16 for r in res]
        for p, q in zip(a.read_grid(lo, size), b.read_grid(lo, size)):
            assert np.array_equal(p, q)
    for s in (a, b):  # a call of several, the grid operator inside g2p
        s._run_substeps(4, a.default_dt)
    sa, sb = a.get_state(), b.get_state()
    for f in sa:
        assert np.array_equal(sa[f], sb[f]), f
