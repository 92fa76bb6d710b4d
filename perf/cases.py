"""The work a user of this framework has it do, as cases that can be timed.

A solver case is one frame of a running simulation: ``step(frame_dt)`` (the
substep count and time step of the solver's own rule) followed by
``particle_info()``, which a program draws or saves.  A batch case is a frame
of an ``MPMSolverBatch``.  A differentiable case is ``DiffMPMSolver.run`` over
some substeps, alone or with its backward pass.

The bodies of a scene are boxes or ellipsoids, each with one material and one
velocity, on a lattice of separate places: they fall, collide and settle while
a case is repeated, as in a program that runs frame after frame.
"""
import math

import numpy as np
import torch

from taichi_elements_amd import MPMSolver, MPMSolverBatch, batch, mpm_solver

WATER, ELASTIC, SNOW, SAND = 0, 1, 2, 3
MATERIALS = {"water": (WATER, ), "mixed": (WATER, ELASTIC, SNOW, SAND),
             "solids": (ELASTIC, SNOW, SAND)}


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------
def _solver(name=None, **kw):
    case = dict(kind="solver", dim=3, res=128, n=1_000_000, bodies=4, frame=1e-2,
                materials="mixed", collider="none", per_cell=8.0, quant=False, g2p2g=False,
                unbounded=False)
    case.update(kw)
    return dict(case, name=name) if name else case


def _batch(name=None, **kw):
    case = dict(kind="batch", dim=3, scenes=16, n=1_000_000, frame=1 / 60, per_cell=8.0)
    case.update(kw)
    return dict(case, name=name) if name else case


def _diff(name=None, **kw):
    case = dict(kind="diff", dim=3, res=128, n=200_000, nsub=16, grad=False, per_cell=8.0)
    case.update(kw)
    return dict(case, name=name) if name else case


def listed():
    return [
        # a 2D teaching scene on a 24^2 grid: the smallest frames there are, all latency
        _solver("water2d_24", dim=2, res=24, n=1_500, bodies=1, frame=8e-3, materials="water",
                per_cell=8.0),
        # the 2D water scene on 128^2
        _solver("water2d_128", dim=2, res=128, n=20_000, bodies=1, frame=8e-3, materials="water",
                per_cell=10.0),
        # a 2D scene for rendering at high resolution, every material, a sphere in the way
        _solver("mixed2d_512", dim=2, res=512, n=400_001, bodies=9, frame=4e-3, per_cell=6.0,
                collider="sphere"),
        # a 3D preview at 64^3, the size at which a scene is set up
        _solver("mixed3d_64", res=64, n=100_003, bodies=5, frame=4e-3),
        # bodies thrown at a sticky ground plane without a box around them (the Blender add-on's mode)
        _solver("unbounded3d_64", res=64, n=50_001, bodies=3, frame=1 / 60, materials="solids",
                collider="sticky", unbounded=True),
        # the main configuration: a million particles of four materials on 128^3, dense
        _solver("mixed3d_128", per_cell=15.0, collider="slip"),
        # the same with packed particle storage
        _solver("quant3d_128", n=777_777, per_cell=8.0, quant=True),
        # the fused transfer
        _solver("g2p2g3d_96", res=96, n=301_003, g2p2g=True),
        # a large sparse domain: sixteen million particles in 64 bodies on 512^3
        _solver("sparse3d_512", res=512, n=16_000_000, bodies=64, frame=2e-3, collider="slip"),
        # many independent scenes together, as for training data
        _batch("batch3d_16", n=1_200_000),
        # a differentiable rollout, forward alone
        _diff("diff_run", nsub=32),
        # and a short one with its gradients, as in an optimisation loop
        _diff("diff_grad", n=150_000, nsub=8, grad=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solver"] * 7 + ["batch"] + ["diff"] * 2)
    if kind == "batch":
        dim = rng.choice([2, 3, 3])
        scenes = rng.randint(2, 16)
        return _batch(dim=dim, scenes=scenes, n=_log_int(rng, 2_000 * scenes, 50_000 * scenes),
                      frame=rng.choice([4e-3, 1e-2, 1 / 60]), per_cell=rng.uniform(4.0, 12.0))
    dim = rng.choice([2, 3, 3])
    if kind == "diff":
        grad = rng.random() < 0.5
        res, per_cell = rng.randint(32, 128), rng.uniform(6.0, 12.0)
        most = min(200_000, (0.15 if dim == 2 else 0.06) * res**dim * per_cell)
        return _diff(dim=dim, res=res, n=_log_int(rng, min(1_000, most), most),
                     nsub=rng.randint(1, 8) if grad else rng.randint(1, 32), grad=grad,
                     per_cell=per_cell)
    mode = rng.choice(["plain"] * 4 + ["quant", "g2p2g", "unbounded"])
    collider = rng.choice(["none", "slip", "sticky", "sphere"])
    frame = rng.choice([2e-3, 4e-3, 8e-3])
    per_cell = rng.uniform(4.0, 16.0)
    if dim == 2:
        res = _log_int(rng, 24, 512)
        most = 0.15 * res * res * per_cell
    else:
        res = _log_int(rng, 24, 256)
        most = min(4_000_000, 0.06 * res**3 * per_cell)
    n = _log_int(rng, min(600, most), most)
    bodies = rng.randint(1, 9) if dim == 2 else rng.randint(1, 16)
    return _solver(dim=dim, res=res, n=n, bodies=bodies, frame=frame, per_cell=per_cell,
                   materials="solids" if mode == "unbounded" else rng.choice(["water", "mixed", "mixed"]),
                   collider="sticky" if mode == "unbounded" else collider,
                   quant=mode == "quant", g2p2g=mode == "g2p2g", unbounded=mode == "unbounded")


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _scene(dim, res, n, bodies, materials, per_cell, seed):
    """Float32 positions and velocities, int32 materials: body k has n // bodies
    particles (the first the rest too) at per_cell particles a cell, a box or an
    ellipsoid, on place k of a lattice that keeps the bodies apart."""
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device=_device())
    gen.manual_seed(int(rng.integers(1 << 40)))
    per_axis = math.ceil(bodies**(1.0 / dim))
    places = rng.permutation(per_axis**dim)[:bodies]
    pitch = 0.88 / per_axis
    xs, vs, ms = [], [], []
    for k in range(bodies):
        count = n // bodies + (n % bodies if k == 0 else 0)
        box = k % 2 == 0
        volume = count / per_cell / res**dim
        aspect = rng.uniform(0.8, 1.25, dim)
        aspect /= np.prod(aspect)**(1.0 / dim)
        ball = {2: math.pi / 4, 3: math.pi / 6}[dim]
        edge = (volume / (1.0 if box else ball))**(1.0 / dim) * aspect
        at = np.array([(places[k] // per_axis**a) % per_axis for a in range(dim)])
        slack = np.maximum(pitch - edge, 0.0)
        centre = 0.06 + at * pitch + edge / 2 + slack * rng.uniform(0.3, 0.7, dim)
        u = torch.rand((count, dim), generator=gen, device=_device()) * 2 - 1
        if not box:  # uniform in the unit ball: directions times a radius
            g = torch.randn((count, dim), generator=gen, device=_device())
            r = torch.rand((count, 1), generator=gen, device=_device())**(1.0 / dim)
            u = g / g.norm(dim=1, keepdim=True) * r
        half = torch.tensor(edge / 2, dtype=torch.float32, device=_device())
        x = torch.tensor(centre, dtype=torch.float32, device=_device()) + u * half
        v = rng.uniform(-0.5, 0.5, dim)
        v[1] = -abs(v[1]) - 0.2
        xs.append(x.cpu().numpy())
        vs.append(np.broadcast_to(v.astype(np.float32), (count, dim)))
        ms.append(np.full(count, MATERIALS[materials][k % len(MATERIALS[materials])], np.int32))
    return np.concatenate(xs), np.concatenate(vs), np.concatenate(ms)


def _gravity(materials, dim):
    """Gentler with snow: it hardens where it is hit, and the explicit time step
    of the solver's default stiffness does not carry a fall from full height."""
    return (0.0, -2.0 if SNOW in MATERIALS[materials] else -9.8, 0.0)[:dim]


COLLIDERS = {
    "slip": ("plane", dict(point=(0.0, 0.05, 0.0), normal=(0.0, 1.0, 0.0), surface=1)),
    "sticky": ("plane", dict(point=(0.0, 0.05, 0.0), normal=(0.1, 1.0, 0.0), surface=0)),
    "sphere": ("sphere", dict(center=(0.5, 0.0, 0.5), radius=0.09, surface=2)),
}


def _collider(case):
    if case["collider"] == "none":
        return None
    kind, kw = COLLIDERS[case["collider"]]
    d = case["dim"]
    return kind, {k: v[:d] if isinstance(v, tuple) else v for k, v in kw.items()}


def _batch_scenes(case, seed):
    """(res, x, v, material) of every scene: uneven sizes, 64^d to 128^d, the
    same for every seed of a case."""
    rng = np.random.default_rng([3, case["n"], case["scenes"]])
    share = np.exp(rng.uniform(0.0, math.log(10.0), case["scenes"]))
    counts = np.maximum(16, (case["n"] * share / share.sum()).astype(int))
    out = []
    for k, n in enumerate(counts):
        res = int(rng.choice([64, 96, 128]))
        n = int(min(n, 0.06 * res**case["dim"] * case["per_cell"]))
        x, v, m = _scene(case["dim"], res, n, int(rng.integers(1, 5)), "mixed", case["per_cell"],
                         [4, seed, k])
        out.append((res, x, v, m))
    return out


def _diff_inputs(case, seed):
    """A state in mid-run: a water body and an elastic one, strained (F within
    5% of the identity) and with a velocity gradient; E per particle."""
    d, n = case["dim"], case["n"]
    x, v, m = _scene(d, case["res"], n, 2, "mixed", case["per_cell"], [5, seed])
    rng = np.random.default_rng([6, seed])
    C = (2.0 * rng.standard_normal((n, d, d))).astype(np.float32)
    F = (np.eye(d) + 0.05 * rng.uniform(-1, 1, (n, d, d))).astype(np.float32)
    Jp = np.ones(n, np.float32)
    water = m == WATER
    F[water] = np.eye(d, dtype=np.float32)
    Jp[water] = rng.uniform(0.97, 1.03, water.sum())
    E = rng.uniform(5e5, 2e6, n).astype(np.float32)
    target = (x.mean(0) + rng.uniform(-0.05, 0.05, d)).astype(np.float32)
    return x, v, C, F, Jp, m, E, target


def prepare(case, seed):
    mpm_solver.PRINT_PROGRESS = batch.PRINT_PROGRESS = False
    d = case["dim"]
    if case["kind"] == "diff":
        from taichi_elements_amd.diff import DiffMPMSolver
        x, v, C, F, Jp, m, E, target = _diff_inputs(case, seed)
        s = DiffMPMSolver((case["res"], ) * d)
        s.setup(m, x)
        state = s.state(x, v)
        n = len(x)
        state[2 * d:2 * d + d * d] = torch.tensor(C.reshape(n, d * d).T.copy(), device=state.device)
        state[2 * d + d * d:2 * d + 2 * d * d] = torch.tensor(F.reshape(n, d * d).T.copy(),
                                                              device=state.device)
        state[-1] = torch.tensor(Jp, device=state.device)
        return dict(case=case, solver=s, state=state, E=torch.tensor(E, device=state.device),
                    nu=torch.tensor(0.2, device=state.device),
                    target=torch.tensor(target, device=state.device))
    if case["kind"] == "batch":
        scenes = _batch_scenes(case, seed)
        b = MPMSolverBatch([dict(res=(res, ) * d) for res, *_ in scenes])
        for s, (_, x, v, m) in zip(b, scenes):
            s.set_gravity(_gravity("mixed", d))
            s.read_restart(len(x), x, v, m, np.full(len(x), 0xFFFFFF, np.int32))
        return dict(case=case, solver=b)
    x, v, m = _scene(d, case["res"], case["n"], case["bodies"], case["materials"],
                     case["per_cell"], [1, seed])
    s = MPMSolver(res=(case["res"], ) * d, quant=case["quant"], use_g2p2g=case["g2p2g"],
                  unbounded=case["unbounded"])
    s.set_gravity(_gravity(case["materials"], d))
    collider = _collider(case)
    if collider:
        getattr(s, {"plane": "add_surface_collider",
                    "sphere": "add_sphere_collider"}[collider[0]])(**collider[1])
    s.read_restart(len(x), x, v, m, np.full(len(x), 0xFFFFFF, np.int32))
    return dict(case=case, solver=s)


def _rows(state, d):
    """What a program reads from a rollout's state.  The rows of C are left out:
    the velocity gradient of a body that moves rigidly is rounding alone."""
    return dict(x=state[0:d], v=state[d:2 * d], F=state[2 * d + d * d:2 * d + 2 * d * d],
                Jp=state[-1])


def run(s):
    case, solver = s["case"], s["solver"]
    if case["kind"] != "diff":
        solver.step(case["frame"])
        return solver.particle_info()
    d = case["dim"]
    if not case["grad"]:
        with torch.no_grad():
            out = solver.run(s["state"], s["E"], s["nu"], case["nsub"], nu_value=0.2)
        return _rows(out, d)
    state = s["state"].clone().requires_grad_(True)
    E = s["E"].clone().requires_grad_(True)
    nu = s["nu"].clone().requires_grad_(True)
    out = solver.run(state, E, nu, case["nsub"], nu_value=0.2)
    loss = _loss(solver.positions(out), out[d:2 * d].T, s["target"])
    loss.backward()
    return dict(_rows(out.detach(), d), grad_x=state.grad[0:d], grad_v=state.grad[d:2 * d],
                grad_F=state.grad[2 * d + d * d:2 * d + 2 * d * d], grad_E=E.grad, grad_nu=nu.grad)


def _loss(x, v, target):
    """Every particle to the target, at rest there."""
    return ((x - target)**2).sum(1).mean() + 0.01 * (v**2).sum(1).mean()


# --------------------------------------------------------------------------
# the work of a pass
# --------------------------------------------------------------------------
def _plan(frame, res):
    """Substep count and dt of step() (a float64 loop that may run one more)."""
    default_dt = 2e-2 / res
    dt = frame / (int(frame / default_dt) + 1)
    left, count = frame, 0
    while left > 0:
        count += 1
        left -= dt
    return count, dt


def _substep_work(d, n, per_cell, quant=False):
    """Bytes and operations of a substep over n particles.  The grid stands
    between p2g and g2p: p2g reads the state and writes F and Jp, g2p reads x
    and writes x, v and C; a node is written and read once by each side."""
    word = 4
    x, C, F = (2, d * d, (d * d + 1) // 2) if quant else (d, d * d, d * d)
    v = 2 if quant else d
    particle = word * ((x + v + C + F + 1 + 1) + (F + 1) + x + (x + v + C))
    nodes = n / per_cell * 1.3
    flops = {2: 500, 3: 2000}[d] * n + 30 * nodes
    return n * particle + nodes * 2 * 4 * (d + 1), flops


def work(case):
    d = case["dim"]
    if case["kind"] == "diff":
        b, f = _substep_work(d, case["n"], case["per_cell"])
        k = case["nsub"] * (3 if case["grad"] else 1)
        return dict(bytes=b * k, flops=f * k)
    read = case["n"] * 4 * (2 * d + 2) * 2  # particle_info: position, velocity, material, colour
    if case["kind"] == "batch":
        count = sum(_plan(case["frame"], r)[0] for r in (64, 96, 128)) / 3
        b, f = _substep_work(d, case["n"], case["per_cell"])
    else:
        count = _plan(case["frame"], case["res"])[0]
        b, f = _substep_work(d, case["n"], case["per_cell"], case["quant"])
    return dict(bytes=b * count + read, flops=f * count)


# --------------------------------------------------------------------------
# the same in 64 bits
# --------------------------------------------------------------------------
class _Exact:
    """MLS-MPM substeps (reference engine/mpm_solver.py:321-735) in float64
    torch: matrices are lists of per-particle vectors."""

    def __init__(self, dim, res, collider=None, unbounded=False, g2p2g=False, E=None, nu=0.2,
                 gravity=-9.8):
        self.gravity = [0.0, gravity, 0.0]
        self.d, self.res, self.dx = dim, res, 1.0 / res
        self.collider, self.unbounded, self.g2p2g = collider, unbounded, g2p2g
        E = 1e6 if E is None else E
        self.mu = E / (2 * (1 + nu))
        self.la = E * nu / ((1 + nu) * (1 - 2 * nu))
        s = math.sin(math.radians(45))
        self.alpha = math.sqrt(2 / 3) * 2 * s / (3 - s)
        self.grid = None

    # small matrices, [i][j] of (n,) tensors
    def mul(self, A, B):
        r = range(self.d)
        return [[sum(A[i][k] * B[k][j] for k in r) for j in r] for i in r]

    def mul_t(self, A, B):
        r = range(self.d)
        return [[sum(A[i][k] * B[j][k] for k in r) for j in r] for i in r]

    def det(self, A):
        if self.d == 2:
            return A[0][0] * A[1][1] - A[0][1] * A[1][0]
        return sum(A[0][j] * (A[1][(j + 1) % 3] * A[2][(j + 2) % 3]
                              - A[1][(j + 2) % 3] * A[2][(j + 1) % 3]) for j in range(3))

    def cof(self, A):
        if self.d == 2:
            return [[A[1][1], -A[1][0]], [-A[0][1], A[0][0]]]
        return [[A[(i + 1) % 3][(j + 1) % 3] * A[(i + 2) % 3][(j + 2) % 3]
                 - A[(i + 1) % 3][(j + 2) % 3] * A[(i + 2) % 3][(j + 1) % 3] for j in range(3)]
                for i in range(3)]

    def polar(self, A, steps=9):
        """The rotation of A by Newton's iteration X <- (X + X^-T) / 2, which
        autograd can follow."""
        X = A
        for _ in range(steps):
            c, det = self.cof(X), self.det(X)
            X = [[0.5 * (X[i][j] + c[i][j] / det) for j in range(self.d)] for i in range(self.d)]
        return X

    def svd(self, A, sweeps=7):
        """U, sigma, V by cyclic Jacobi rotations of A^T A (det A > 0)."""
        d = self.d
        S = [[sum(A[k][i] * A[k][j] for k in range(d)) for j in range(d)] for i in range(d)]
        one, zero = torch.ones_like(A[0][0]), torch.zeros_like(A[0][0])
        V = [[one if i == j else zero for j in range(d)] for i in range(d)]
        for _ in range(sweeps):
            for p, q in ((0, 1), (0, 2), (1, 2)) if d == 3 else ((0, 1), ):
                diff, off = S[q][q] - S[p][p], S[p][q]
                den = diff.abs() + torch.sqrt(diff * diff + 4 * off * off)
                t = torch.where(den > 0, 2 * off / torch.where(den > 0, den, one), zero)
                t = torch.where(diff >= 0, t, -t)
                c = 1 / torch.sqrt(1 + t * t)
                s = c * t
                for M in (S, V):
                    for k in range(d):
                        M[k][p], M[k][q] = c * M[k][p] - s * M[k][q], s * M[k][p] + c * M[k][q]
                for k in range(d):
                    S[p][k], S[q][k] = c * S[p][k] - s * S[q][k], s * S[p][k] + c * S[q][k]
        B = self.mul(A, V)
        sig = [torch.sqrt(sum(B[i][j]**2 for i in range(d))) for j in range(d)]
        return [[B[i][j] / sig[j] for j in range(d)] for i in range(d)], sig, V

    def constitutive(self, m, F, C, Jp, dt):
        """(F, Jp, Kirchhoff stress) after the trial step (I + dt C) F."""
        d = self.d
        r = range(d)
        water = m == WATER
        if not self.g2p2g:
            F = [[torch.where(water, Jp if i == j == 0 else torch.full_like(Jp, float(i == j)), F[i][j])
                  for j in r] for i in r]
        F = self.mul([[float(i == j) + dt * C[i][j] for j in r] for i in r], F)
        J = self.det(F)
        snow, sand, elastic = m == SNOW, m == SAND, m == ELASTIC
        h = torch.where(snow, torch.exp(10 * (1 - Jp)), torch.ones_like(Jp))
        if self.g2p2g:
            h = torch.where(water, torch.exp(10 * (1 - Jp)), h)
        h = torch.where(elastic, torch.full_like(h, 0.3), h)
        if bool((snow | sand).any()):
            U, sig, V = self.svd(F)
            R = self.mul_t(U, V)
            clamped = [torch.clamp(s, 1 - 2.5e-2, 1 + 4.5e-3) for s in sig]
            eps = [torch.log(torch.clamp(s, min=1e-4)) for s in sig]
            tr = sum(eps) + Jp
            hat = [e - tr / d for e in eps]
            norm = torch.sqrt(sum(e * e for e in hat)) + 1e-20
            gamma = norm + (d * self.la + 2 * self.mu) / (2 * self.mu) * tr * self.alpha
            k = torch.clamp(gamma, min=0) / norm
            proj = [torch.where(tr >= 0, torch.ones_like(tr), torch.exp(e - k * f))
                    for e, f in zip(eps, hat)]
            new = [torch.where(sand, b, torch.where(snow, a, s))
                   for a, b, s in zip(clamped, proj, sig)]
            ratio = 1
            for s, c in zip(sig, clamped):
                ratio = ratio * s / c
            Jp_new = torch.where(snow, Jp * ratio,
                                 torch.where(sand, torch.where(tr >= 0, tr, torch.zeros_like(tr)), Jp))
            plastic = snow | sand
            Fp = self.mul_t([[U[i][j] * new[j] for j in r] for i in r], V)
            F = [[torch.where(plastic, Fp[i][j], F[i][j]) for j in r] for i in r]
            J = torch.where(plastic, self.det(F), J)
            logs = [torch.log(s) for s in new]
            centre = [(2 * self.mu * l + self.la * sum(logs)) / s for l, s in zip(logs, new)]
            T = self.mul_t(self.mul_t([[U[i][j] * centre[j] for j in r] for i in r], V), F)
        else:
            # water takes no part in the rotation (its mu is 0)
            R = self.polar([[torch.where(water, torch.full_like(Jp, float(i == j)), F[i][j])
                             for j in r] for i in r])
            Jp_new, T = Jp, None
        F = [[torch.where(water, J if i == j == 0 else torch.full_like(Jp, float(i == j)), F[i][j])
              for j in r] for i in r]
        if not self.g2p2g:
            Jp_new = torch.where(water, J, Jp_new)
        mu = torch.where(water, torch.zeros_like(h), h * self.mu)
        stress = self.mul_t([[2 * mu * (F[i][j] - R[i][j]) for j in r] for i in r], F)
        iso = h * self.la * J * (J - 1)
        stress = [[stress[i][j] + (iso if i == j else 0) for j in r] for i in r]
        if T is not None:
            stress = [[torch.where(sand, T[i][j], stress[i][j]) for j in r] for i in r]
        return F, Jp_new, stress

    def stencil(self, x):
        t = [c * self.res for c in x]
        base = [torch.floor(c.detach() - 0.5) for c in t]
        fx = [c - b for c, b in zip(t, base)]
        w = [[0.5 * (1.5 - f)**2, 0.75 - (f - 1)**2, 0.5 * (f - 0.5)**2] for f in fx]
        return [b.long() for b in base], fx, w

    def nodes(self, base, fx, w):
        """(flat index, weight, node - x in cells) of every stencil node."""
        d = self.d
        for k in range(3**d):
            o = [(k // 3**a) % 3 for a in range(d)]
            idx, wt = 0, 1
            for a in reversed(range(d)):
                idx = idx * self.extent[a] + (base[a] + (o[a] - self.lo[a]))
            for a in range(d):
                wt = wt * w[a][o[a]]
            yield idx, wt, [o[a] - fx[a] for a in range(d)]

    def scatter(self, x, v, C, stress, mass, dt):
        d = self.d
        base, fx, w = self.stencil(x)
        ends = torch.stack([torch.stack([b.min(), b.max()]) for b in base]).tolist()
        self.lo = [int(e[0]) for e in ends]
        self.extent = [int(e[1]) - int(e[0]) + 3 for e in ends]
        scale = -dt * self.dx**d * 4 * self.res**2
        A = [[(scale * stress[i][j] + mass * C[i][j]) * self.dx for j in range(d)] for i in range(d)]
        size = math.prod(self.extent)
        # one column a channel: momentum, mass
        cols = [torch.zeros(size, dtype=mass.dtype, device=mass.device) for _ in range(d + 1)]
        for idx, wt, dp in self.nodes(base, fx, w):
            for i in range(d):
                c = wt * (mass * v[i] + sum(A[i][j] * dp[j] for j in range(d)))
                cols[i] = cols[i].index_add(0, idx, c) if c.requires_grad else cols[i].index_add_(0, idx, c)
            c = wt * mass
            cols[d] = cols[d].index_add(0, idx, c) if c.requires_grad else cols[d].index_add_(0, idx, c)
        return cols

    def grid_op(self, cols, dt):
        d, m = self.d, cols[self.d]
        full = m > 0
        inv = torch.where(full, 1 / torch.where(full, m, torch.ones_like(m)), torch.zeros_like(m))
        v = [cols[a] * inv + torch.where(full, dt * self.gravity[a], 0.0) for a in range(d)]
        if self.g2p2g:
            most = self.dx * 0.9 / dt
            v = [torch.clamp(c, -most, most) for c in v]
        flat = torch.arange(m.numel(), device=m.device)
        I = []
        for a in range(d):
            I.append(flat % self.extent[a] + self.lo[a])
            flat = flat // self.extent[a]
        lo, hi = (-2048 + 3, 2048 - 3) if self.unbounded else (3, self.res - 3)
        for a in range(d):
            stop = ((I[a] < lo) & (v[a] < 0)) | ((I[a] >= hi) & (v[a] > 0))
            v[a] = torch.where(stop, torch.zeros_like(v[a]), v[a])
        if self.collider:
            kind, kw = self.collider
            at = kw["point"] if kind == "plane" else kw["center"]
            off = [I[a] * self.dx - at[a] for a in range(d)]
            if kind == "plane":
                length = math.sqrt(sum(c * c for c in kw["normal"]))
                normal = [c / length for c in kw["normal"]]
                inside = sum(o * c for o, c in zip(off, normal)) < 0
            else:
                r = torch.sqrt(sum(o * o for o in off))
                normal = [o / (r + 1e-5) for o in off]
                inside = r < kw["radius"]
            vn = sum(c * u for c, u in zip(normal, v))
            if kw["surface"] == 0:
                new = [torch.zeros_like(c) for c in v]
            else:
                take = vn if kw["surface"] == 1 else torch.clamp(vn, max=0)
                new = [u - c * take for c, u in zip(normal, v)]
            v = [torch.where(inside, b, a) for a, b in zip(v, new)]
        return v

    def gather(self, x, grid):
        d = self.d
        base, fx, w = self.stencil(x)
        v, C = [0] * d, [[0] * d for _ in range(d)]
        for idx, wt, dp in self.nodes(base, fx, w):
            for i in range(d):
                u = wt * grid[i][idx]
                v[i] = v[i] + u
                for j in range(d):
                    C[i][j] = C[i][j] + 4 * self.res * u * dp[j]
        return v, C

    def substep(self, x, v, C, F, Jp, m, dt):
        if self.g2p2g:  # gather, move, update, scatter at the new place
            if self.grid is not None:
                v, C = self.gather(x, self.grid)
            x = [a + dt * b for a, b in zip(x, v)]
            F, Jp, stress = self.constitutive(m, F, C, Jp, dt)
            mass = torch.full_like(x[0], self.dx**self.d * 1000)
            self.grid = self.grid_op(self.scatter(x, v, C, stress, mass, dt), dt)
            return x, v, C, F, Jp
        F, Jp, stress = self.constitutive(m, F, C, Jp, dt)
        mass = torch.full_like(x[0], self.dx**self.d * 1000)
        grid = self.grid_op(self.scatter(x, v, C, stress, mass, dt), dt)
        v, C = self.gather(x, grid)
        return [a + dt * b for a, b in zip(x, v)], v, C, F, Jp


def _columns(a):
    return [torch.tensor(a[:, k].astype(np.float64), device=_device()) for k in range(a.shape[1])]


def _frame_exact(case, res, x, v, m):
    d = case["dim"]
    collider = _collider(case) if "collider" in case else None
    e = _Exact(d, res, collider, case.get("unbounded", False), case.get("g2p2g", False),
               gravity=_gravity(case.get("materials", "mixed"), d)[1])
    count, dt = _plan(case["frame"], res)
    x, v, m = _columns(x), _columns(v), torch.tensor(m, device=_device())
    zero, one = torch.zeros_like(x[0]), torch.ones_like(x[0])
    C = [[zero for _ in range(d)] for _ in range(d)]
    F = [[one if i == j else zero for j in range(d)] for i in range(d)]
    Jp = torch.where(m == SAND, zero, one)
    for _ in range(count):
        x, v, C, F, Jp = e.substep(x, v, C, F, Jp, m, dt)
    return dict(position=torch.stack(x, 1).cpu().numpy(), velocity=torch.stack(v, 1).cpu().numpy(),
                material=None, color=None)


def exact(case, seed):
    d = case["dim"]
    if case["kind"] == "solver":
        # packed storage rounds the state after every substep; and the largest take too long
        if case["quant"] or case["n"] * _plan(case["frame"], case["res"])[0] > 70_000_000:
            return None
        x, v, m = _scene(d, case["res"], case["n"], case["bodies"], case["materials"],
                         case["per_cell"], [1, seed])
        return _frame_exact(case, case["res"], x, v, m)
    if case["kind"] == "batch":
        return [_frame_exact(case, *s) for s in _batch_scenes(case, seed)]
    x, v, C, F, Jp, m, E, target = _diff_inputs(case, seed)
    grad = case["grad"]
    leaf = lambda t: t.requires_grad_(grad)  # noqa: E731
    x, v = [leaf(c) for c in _columns(x)], [leaf(c) for c in _columns(v)]
    n = len(m)
    Cc = _columns(C.reshape(n, d * d))
    Fc = [leaf(c) for c in _columns(F.reshape(n, d * d))]
    Jp = torch.tensor(Jp.astype(np.float64), device=_device())
    E = leaf(torch.tensor(E.astype(np.float64), device=_device()))
    nu = leaf(torch.tensor(0.2, dtype=torch.float64, device=_device()))
    m = torch.tensor(m, device=_device())
    e = _Exact(d, case["res"], E=E, nu=nu)
    y, u, M, G = x, v, [Cc[i * d:i * d + d] for i in range(d)], [Fc[i * d:i * d + d] for i in range(d)]
    for _ in range(case["nsub"]):
        y, u, M, G, Jp = e.substep(y, u, M, G, Jp, m, 2e-2 / case["res"])
    cells = [c for row in G for c in row]
    out = dict(x=torch.stack(y).detach(), v=torch.stack(u).detach(),
               F=torch.stack(cells).detach(), Jp=Jp.detach())
    if grad:
        target = torch.tensor(target.astype(np.float64), device=_device())
        _loss(torch.stack(y, 1), torch.stack(u, 1), target).backward()
        zero = torch.zeros_like(Jp.detach())
        rows = lambda a: torch.stack([c.grad if c.grad is not None else zero for c in a])  # noqa: E731
        out.update(grad_x=rows(x), grad_v=rows(v), grad_F=rows(Fc), grad_E=E.grad, grad_nu=nu.grad)
    return {k: t.cpu().numpy() for k, t in out.items()}
