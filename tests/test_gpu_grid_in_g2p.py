"""The grid operator inside g2p (small scenes, every substep of a call but
the last) against the grid operator kernel (a call of one substep): the sums
take the same order, so state and grid are bitwise the same."""
import numpy as np
import pytest

from tests.helpers import cube_particles

pytestmark = pytest.mark.gpu

LINE = 160 * 1024  # particles up to which g2p runs the grid operator


@pytest.fixture(autouse=True)
def _quiet():
    from taichi_elements_amd import batch, mpm_solver
    mpm_solver.PRINT_PROGRESS = batch.PRINT_PROGRESS = False


def _scene(dim, res, n, chunk, **options):
    from taichi_elements_amd import MPMSolver
    rng = np.random.default_rng(n + chunk)
    s = MPMSolver(res=(res, ) * dim, chunk=chunk, **options)
    s.add_sphere_collider([0.5] * dim, 0.1, s.surface_slip)
    s.add_surface_collider([0.0, 0.3, 0.0][:dim], [0.1, 1.0, 0.0][:dim], s.surface_separate, 0.2)
    x = cube_particles(rng, n, [0.02] * dim, [0.6] * dim, dim)
    s.read_restart(n, x, rng.uniform(-1, 1, (n, dim)).astype(np.float32),
                   rng.integers(0, 5, n).astype(np.int32), np.zeros(n, np.int32))
    return s


@pytest.mark.parametrize("dim,res,n,chunk,options", [
    (2, 16, 1, 256, {}),
    (2, 33, 3000, 16, {}),
    (2, 48, 20000, 1024, dict(quant=True)),
    (2, 128, LINE, 256, {}),
    (2, 128, LINE + 1, 256, {}),
    (3, 16, 1, 256, {}),
    (3, 24, 20000, 64, {}),
    (3, 32, 9001, 1024, dict(quant=True)),
    (3, 96, LINE, 256, {}),
    (3, 96, LINE + 1, 256, {}),
    # more chunks than it is taken for, known after the first call
    (2, 128, 60000, 16, {}),
    (3, 48, 60000, 16, {}),
])
def test_call_of_many_substeps_is_bitwise_single_substeps(dim, res, n, chunk, options):
    a, b = (_scene(dim, res, n, chunk, **options) for _ in range(2))
    for count in (5, 1, 3):
        a._run_substeps(count, a.default_dt)
        for _ in range(count):
            b._run_substeps(1, b.default_dt)
        sa, sb = a.get_state(), b.get_state()
        for k in sa:
            assert np.array_equal(sa[k], sb[k]), (count, k)
        lo, size = [-8] * dim, [res + 16] * dim
        for p, q in zip(a.read_grid(lo, size), b.read_grid(lo, size)):
            assert np.array_equal(p, q)


@pytest.mark.parametrize("dim", [2, 3])
def test_scenes_that_sit_out(dim):
    """A batch of scenes, one of which sits the call out: it keeps its
    state, the others advance as alone."""
    from taichi_elements_amd import MPMSolver, MPMSolverBatch
    rng = np.random.default_rng(5)
    parts = []
    for k in range(3):
        n = 1500 + 700 * k
        parts.append((cube_particles(rng, n, [0.2] * dim, [0.4, 0.3, 0.4][:dim], dim),
                      rng.uniform(-1, 1, (n, dim)).astype(np.float32),
                      rng.integers(0, 4, n).astype(np.int32)))
    b = MPMSolverBatch([dict(res=(24 + 8 * k, ) * dim) for k in range(3)])
    solos = [MPMSolver(res=(24 + 8 * k, ) * dim) for k in range(3)]
    for s, t, (x, v, m) in zip(b, solos, parts):
        for u in (s, t):
            u.read_restart(len(x), x, v, m, np.zeros(len(x), np.int32))
    dts = b.default_dts()
    for calls, out in ((4, None), (20, 1), (3, None)):
        b.substeps(calls, [0.0 if k == out else dt for k, dt in enumerate(dts)])
        for k, (t, dt) in enumerate(zip(solos, dts)):
            if k != out:
                t._run_substeps(calls, dt)
    for s, t in zip(b, solos):
        got, ref = s.get_state(), t.get_state()
        for k in got:
            assert np.array_equal(got[k], ref[k]), k
