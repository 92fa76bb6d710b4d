"""Who owns the arrays that a batch's readers return: a scene's own
particle_info() holds no more than that scene's particles; the batch's may share
its memory between scenes, but no two of them overlap."""
import numpy as np
import pytest

from tests.helpers import cube_particles

pytestmark = pytest.mark.gpu


def test_particle_info_arrays():
    from taichi_elements_amd import MPMSolverBatch, batch, mpm_solver
    mpm_solver.PRINT_PROGRESS = batch.PRINT_PROGRESS = False
    rng = np.random.default_rng(1)
    b = MPMSolverBatch([dict(res=(32, ) * 3) for _ in range(3)])
    xs = [cube_particles(rng, n, [0.2] * 3, [0.5] * 3, 3) for n in (500, 700, 1)]
    for s, x in zip(b, xs):
        s.add_particles(x, 1)
    for s, x in zip(b, xs):
        info = s.particle_info()
        assert np.array_equal(info["position"], x)
        for a in info.values():
            assert a.base is None and a.flags.owndata and a.flags.writeable
            assert a.flags.c_contiguous
    every = b.particle_info()
    for i, info in enumerate(every):
        for k, a in info.items():
            assert a.flags.writeable and a.flags.c_contiguous
            for other in every[i + 1:]:
                assert not np.shares_memory(a, other[k])
