"""DiffMPMSolver's particle reordering: the kernel moves float32 words and
computes nothing, so every result is bitwise that of torch indexing -- for
few and many rows (the kernel deals eight rows at a time out to the XCDs),
any column count, and strided, transposed and expanded inputs -- and a run
keeps no record of its substeps when no gradient is asked for."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import torch  # noqa: E402


def _solver(n, seed=3):
    from taichi_elements_amd.diff import DiffMPMSolver
    ds = DiffMPMSolver((32, 32, 32))
    rng = np.random.default_rng(seed)
    x = rng.uniform(0.3, 0.7, (n, 3)).astype(np.float32)
    ds.setup(rng.integers(0, 2, n).astype(np.int32), x)
    return ds, x


@pytest.mark.parametrize("n", [1, 63, 257, 5001, 300_001])
@pytest.mark.parametrize("rows", [0, 1, 7, 8, 9, 13, 25])
def test_reordering_is_indexing(n, rows):
    from taichi_elements_amd.diff import _Reorder
    ds, _ = _solver(n)
    base = torch.randn(max(rows, 1), 2 * n, device=ds.device)
    views = [base[:rows, :n], base[:rows, ::2], base[:rows].T.contiguous().T[:, :n],
             base[:1, :n].expand(rows, n), base[0, :n], base[0, ::2]]
    for t in views:
        t = t.detach().requires_grad_()
        got = _Reorder.apply(t, ds, ds._order, ds._inverse)
        ref = t[..., ds._order]
        assert got.is_contiguous() and torch.equal(got, ref)
        g = torch.randn_like(ref)
        for cot in (g, g.T.contiguous().T if g.dim() == 2 else g, g[..., :1].expand(g.shape)):
            a, = torch.autograd.grad(got, t, cot, retain_graph=True)
            b, = torch.autograd.grad(ref, t, cot, retain_graph=True)
            assert torch.equal(a, b)


def test_run_without_gradients_is_the_run_with_them():
    ds, x = _solver(3000)
    s0 = ds.state(x)
    E = torch.full((3000, ), 1e6, device=ds.device)
    nu = torch.tensor(0.2, device=ds.device)
    plain = ds.run(s0, E, nu, 5)
    ds.check()
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    kept = ds.run(s0, E.clone().requires_grad_(), nu, 5)
    torch.cuda.synchronize()
    assert torch.cuda.memory_allocated() - before > 5 * ds._binning_bytes
    assert torch.equal(plain, kept.detach())
    with torch.no_grad():
        assert torch.equal(plain, ds.run(s0, E.clone().requires_grad_(), nu, 5))
    # no substeps: indexing there and back, in any dtype
    assert torch.equal(ds.run(s0, E, nu, 0), s0)
    assert torch.equal(ds.run(s0.double(), E, nu, 0), s0.double())
