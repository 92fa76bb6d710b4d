"""DiffMPMSolver.run on lazily negated views (the imaginary part of a conjugate,
real tensors with the negative bit set): the particle reordering reads raw
memory, indexing does not.  Outputs and gradients are bitwise those of the same
values laid out plainly, as inputs and as the cotangent."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import torch  # noqa: E402


def _negated(t):
    """The values of t as a view whose memory holds -t."""
    z = torch.complex(torch.zeros_like(t), -t).conj().imag
    assert z.is_neg() and torch.equal(z, t)
    return z


@pytest.mark.parametrize("n", [1, 700])
def test_negated_views(n):
    from taichi_elements_amd.diff import DiffMPMSolver, _Reorder
    ds = DiffMPMSolver((32, 32, 32))
    rng = np.random.default_rng(n)
    x = rng.uniform(0.3, 0.7, (n, 3)).astype(np.float32)
    ds.setup(rng.integers(0, 2, n).astype(np.int32), x)
    s0 = ds.state(x, rng.uniform(-1, 1, (n, 3)).astype(np.float32))
    E = torch.full((n, ), 1e6, device=ds.device)
    nu = torch.tensor(0.2, device=ds.device)

    def run(state, youngs):
        out = ds.run(state, youngs, nu, 3)
        ds.check()
        return out

    ref = run(s0, E)
    assert torch.equal(run(_negated(s0), E), ref)
    assert torch.equal(run(s0, _negated(E)), ref)

    def grads(state, youngs, wrap):
        a, e = state.clone().requires_grad_(), youngs.clone().requires_grad_()
        return torch.autograd.grad(run(wrap(a), wrap(e)), (a, e), s0)

    plain = grads(s0, E, lambda t: t)
    for a, b in zip(grads(s0, E, lambda t: torch.complex(torch.zeros_like(t), -t).conj().imag),
                    plain):
        assert torch.equal(a, b)
    t = torch.randn(25, n, device=ds.device, requires_grad=True)
    cot = _negated(torch.randn(25, n, device=ds.device))
    a, = torch.autograd.grad(_Reorder.apply(t, ds, ds._order, ds._inverse), t, cot)
    b, = torch.autograd.grad(t[:, ds._order], t, cot)
    assert torch.equal(a, b)
