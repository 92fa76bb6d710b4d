"""Differentiable substeps recorded in a HIP graph, replayed between eager ones:
the handle's block counts start from zero in each, whatever ran before.  The
graph holds a substep and the backward that bins again (no record), or two such
backwards: an even number of binnings, so the double buffers are in step with
the eager calls.  Every output is compared bitwise with the first one."""
import ctypes

import numpy as np
import pytest

from tests.helpers import cube_particles, deformed_state

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("substep_in_graph", [True, False])
def test_replays_between_eager_substeps(dim, substep_in_graph):
    from taichi_elements_amd import _lib
    from taichi_elements_amd._lib import check
    from taichi_elements_amd.diff import DiffMPMSolver, _ptr, _stream
    L = _lib.lib()
    rng = np.random.default_rng(5)
    n = 3001
    x = cube_particles(rng, n, [0.3] * dim, [0.35] * dim, dim)
    mat = rng.integers(0, 4, n).astype(np.int32)
    st = deformed_state(rng, x, mat, dim)
    ds = DiffMPMSolver((32, ) * dim)
    ds.setup(mat)
    rows = [st["x"].T, st["v"].T, st["C"].reshape(n, dim * dim).T,
            st["F"].reshape(n, dim * dim).T, st["Jp"][None]]
    s0 = torch.tensor(np.ascontiguousarray(np.concatenate(rows, 0), np.float32),
                      device=ds.device)
    E = torch.tensor(rng.uniform(5e5, 2e6, n).astype(np.float32), device=ds.device)
    g = torch.randn_like(s0)
    dt = ctypes.c_float(ds.default_dt)

    def forward(out):
        check(L.mpm_diff_substep(ds._handle, dt, _ptr(s0), _ptr(out), _ptr(E), 0.2, None,
                                 _stream()))

    def backward(grads):
        check(L.mpm_diff_substep_backward(ds._handle, dt, _ptr(s0), _ptr(E), 0.2, None, _ptr(g),
                                          _ptr(grads[0]), _ptr(grads[1]), _ptr(grads[2]),
                                          _stream()))

    def empty_grads():
        return torch.empty_like(s0), torch.empty_like(E), torch.empty(1, device=ds.device)

    ref, ref_grads = torch.empty_like(s0), empty_grads()
    forward(ref)
    backward(ref_grads)
    ds.check()

    out, grads = torch.empty_like(s0), empty_grads()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        if substep_in_graph:
            forward(out)
        else:
            backward(grads)
        backward(grads)
    for eager in (0, 2, 2, 4, 2):
        for t in (out, *grads):
            t.fill_(float("nan"))
        graph.replay()
        ds.check()
        assert torch.equal(out, ref) or not substep_in_graph
        for a, b in zip(grads, ref_grads):
            assert torch.equal(a, b)
        for _ in range(eager):
            again = torch.full_like(s0, float("nan"))
            forward(again)
            ds.check()
            assert torch.equal(again, ref)
