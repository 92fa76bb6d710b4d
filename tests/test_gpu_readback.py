"""particle_info() and get_state() through the pinned slots: sizes of one
slot, of several, and around a slot's end, read several times; every storage
mode; a batch's scenes as views and as copies."""
import numpy as np
import pytest

from tests.helpers import cube_particles

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _quiet():
    from taichi_elements_amd import batch, mpm_solver
    mpm_solver.PRINT_PROGRESS = batch.PRINT_PROGRESS = False


@pytest.mark.parametrize("dim,n,options", [
    (2, 1, {}),
    (2, 104857, {}),   # 20 bytes a particle (x, v, material): just below one 2 MiB slot
    (2, 104858, {}),   # and just above
    (3, 74898, {}),    # 28 bytes a particle: the same
    (3, 74899, {}),
    (3, 700001, {}),   # several slots in turn
    (3, 150000, dict(quant=True)),
    (3, 30000, dict(quant=True, use_g2p2g=True, support_plasticity=False)),
])
def test_readers_agree_with_what_was_set(dim, n, options):
    from taichi_elements_amd import MPMSolver
    rng = np.random.default_rng(n)
    x = cube_particles(rng, n, [0.1] * dim, [0.8] * dim, dim)
    v = rng.uniform(-1, 1, (n, dim)).astype(np.float32)
    m = rng.integers(0, 5, n).astype(np.int32)
    col = rng.integers(0, 1 << 24, n).astype(np.int32)
    s = MPMSolver(res=(64, ) * dim, **options)
    s.read_restart(n, x, v, m, col)
    first = None
    for _ in range(4):  # the first read takes another way than the later ones
        info = s.particle_info()
        got = s.get_state()
        for a, b in (("position", "x"), ("velocity", "v"), ("material", "material"),
                     ("color", "color")):
            assert np.array_equal(info[a], got[b]), a
        assert np.array_equal(info["material"], m) and np.array_equal(info["color"], col)
        if not options:
            assert np.array_equal(info["position"], x) and np.array_equal(info["velocity"], v)
        else:  # the packed formats' steps
            assert np.abs(info["position"] - x).max() <= 2.0**-19
            assert np.abs(info["velocity"] - v).max() <= 2.0**-18
        first = first or info
        for k in info:
            assert np.array_equal(info[k], first[k])


def test_scenes_of_a_batch():
    from taichi_elements_amd import MPMSolverBatch
    rng = np.random.default_rng(3)
    b = MPMSolverBatch([dict(res=(32, ) * 3), dict(res=(40, ) * 3)])
    xs = [cube_particles(rng, n, [0.2] * 3, [0.5] * 3, 3) for n in (500, 700, 300)]
    b[0].add_particles(xs[0], 1)
    b[1].add_particles(xs[1], 2)
    b[0].add_particles(xs[2], 3)  # scene 0 in two runs, scene 1 in one
    info = b.particle_info()
    assert np.array_equal(info[0]["position"], np.concatenate([xs[0], xs[2]]))
    assert np.array_equal(info[1]["position"], xs[1])
    assert np.array_equal(b[1].particle_info()["position"], xs[1])
    info[1]["position"][:] = 0  # the caller's own memory
    assert np.array_equal(b[1].particle_info()["position"], xs[1])
