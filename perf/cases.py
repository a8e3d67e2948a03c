"""The workloads that this framework's speed is judged by, as a user's program
runs them through ``GLSolver``, ``BatchTD`` and ``BatchCG``.

A case is a plain dict. Kinds:

td        time-dependent run: ``gl.solve.td(dt=0.1, Nt=steps)`` from a given state
cg        minimisation: ``gl.solve.cg(n_iter=steps)``, then the free energy
batch_td  independent instances of mixed sizes advanced together (BatchTD)
batch_cg  independent instances minimised together (BatchCG)
analysis  everything read off a state: free energy, B, J, J_s, vortices

Common fields: Nx, Ny (nodes), dtype ('float32' / 'float64'), kappa (0 stands
for infinity: A is fixed), disorder (a material mask with holes; for the time
evolution and the analysis a pinning map eps(r) too), steps. Grid spacing 0.5,
conductivity 200, field H = 0.1.

States look like developed ones: a smooth order parameter with vortices
(|psi| <= 1), the vector potential of the field plus a smooth screening part.
Every pass starts from that state: it is copied back, device to device, first.
"""
import math

import numpy as np
import torch

from svirl_amd import GLSolver
from svirl_amd.batch import BatchCG, BatchTD

DX = 0.5
DT = 0.1
SIGMA = 200.0
H = 0.1
STOP = 1e-6            # GLSolver's default stop criteria of both Jacobi solves


def listed():
    return [
        # the smallest production grid: film in the kappa = inf limit, the default precision
        dict(name="td_129_f64", kind="td", Nx=129, Ny=129, dtype="float64", kappa=0.0, disorder=False, steps=20),
        # a small sample with holes and pinning, screening on, odd sides
        dict(name="td_97x203_f32", kind="td", Nx=97, Ny=203, dtype="float32", kappa=5.0, disorder=True, steps=20),
        # the middle of the range: a clean square sample with screening
        dict(name="td_1025_f32", kind="td", Nx=1025, Ny=1025, dtype="float32", kappa=5.0, disorder=False, steps=20),
        # a ragged sample of that size in the default precision
        dict(name="td_771x1283_f64", kind="td", Nx=771, Ny=1283, dtype="float64", kappa=5.0, disorder=True, steps=10),
        # the large disordered film that the framework's headline is quoted on, both precisions
        dict(name="td_4097_f32", kind="td", Nx=4097, Ny=4097, dtype="float32", kappa=5.0, disorder=True, steps=10),
        dict(name="td_4097_f64", kind="td", Nx=4097, Ny=4097, dtype="float64", kappa=5.0, disorder=True, steps=4),
        # a quick minimisation of a small film
        dict(name="cg_129_f32", kind="cg", Nx=129, Ny=129, dtype="float32", kappa=0.0, disorder=False, steps=20),
        # the default precision, whose line search runs on the host
        dict(name="cg_1025_f64", kind="cg", Nx=1025, Ny=1025, dtype="float64", kappa=5.0, disorder=False, steps=10),
        # minimisation of the large film
        dict(name="cg_4097_f32", kind="cg", Nx=4097, Ny=4097, dtype="float32", kappa=5.0, disorder=True, steps=10),
        # a parameter scan: 32 samples of 65 to 1025 nodes a side at once
        dict(name="batch_td_32_f32", kind="batch_td", count=32, Nx=1025, Ny=1025, dtype="float32", kappa=5.0,
             disorder=True, steps=10),
        # many equal samples relaxed at once
        dict(name="batch_cg_256x129_f32", kind="batch_cg", count=256, Nx=129, Ny=129, dtype="float32", kappa=5.0,
             disorder=True, steps=8),
        # what a program reads off a state between runs
        dict(name="analysis_1000x1501_f32", kind="analysis", Nx=1000, Ny=1501, dtype="float32", kappa=5.0,
             disorder=True, steps=1),
    ]


def _side(rng, lo, hi):
    """A number of nodes, spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["td", "td", "td", "cg", "cg", "batch_td", "batch_cg", "analysis"])
    c = dict(kind=kind, dtype=rng.choice(["float32", "float64"]), kappa=rng.choice([0.0, 2.0, 5.0]),
             disorder=rng.random() < 0.5)
    wide = c["dtype"] == "float64"
    if kind == "td":
        c["Nx"], c["Ny"] = _side(rng, 33, 4097), _side(rng, 33, 4097)
        c["steps"] = rng.randint(1, 4) if c["Nx"] * c["Ny"] > 4e6 else rng.randint(1, 20)
    elif kind == "cg":
        c["Nx"], c["Ny"] = _side(rng, 33, 2900 if wide else 4097), _side(rng, 33, 2900 if wide else 4097)
        c["steps"] = rng.randint(2, 10)
    elif kind == "batch_td":
        c["count"] = rng.randint(4, 32)
        c["Nx"], c["Ny"] = _side(rng, 65, 1025), _side(rng, 65, 1025)  # the largest sides of the batch
        c["steps"] = rng.randint(2, 10)
    elif kind == "batch_cg":
        c["Nx"], c["Ny"] = _side(rng, 33, 257), _side(rng, 33, 257)
        c["count"] = max(8, min(256, int(4.3e6 / (c["Nx"] * c["Ny"]))))
        c["steps"] = rng.randint(2, 8)
        c["kappa"] = rng.choice([2.0, 5.0])
    else:
        c["Nx"], c["Ny"] = _side(rng, 65, 2049), _side(rng, 65, 2049)
        c["steps"] = 1
    return c


# ---------------------------------------------------------------- inputs

def _smooth(shape, gen, sigma=4):
    """Unit-variance Gaussian noise of correlation length `sigma` grid steps, periodic."""
    f = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
    r = 3 * sigma
    w = [math.exp(-0.5 * (k / sigma) ** 2) for k in range(-r, r + 1)]
    n = math.sqrt(sum(v * v for v in w))
    for axis in (0, 1):
        f = sum(torch.roll(f, k, axis) * (w[k + r] / n) for k in range(-r, r + 1))
    return f


def _fields(Nx, Ny, kappa, disorder, dtype, seed, pinned):
    """psi (Ny, Nx), a (Ny, Nx-1), b (Ny-1, Nx), material cells or None, eps map or None,
    on the GPU and already rounded to `dtype`."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    real = torch.float32 if dtype == "float32" else torch.float64
    z = torch.complex(_smooth((Ny, Nx), gen), _smooth((Ny, Nx), gen))
    m = z.abs().clamp_min(1e-12)
    psi = z / m * torch.tanh(1.5 * m)
    Lx, Ly = DX * (Nx - 1), DX * (Ny - 1)
    y = torch.arange(Ny, device="cuda", dtype=torch.float64) * DX
    x = torch.arange(Nx, device="cuda", dtype=torch.float64) * DX
    a = (-0.5 * H * (y - 0.5 * Ly))[:, None].repeat(1, Nx - 1)
    b = (0.5 * H * (x - 0.5 * Lx))[None, :].repeat(Ny - 1, 1)
    if kappa:
        a = a + 0.02 * _smooth((Ny, Nx - 1), gen, 8)
        b = b + 0.02 * _smooth((Ny - 1, Nx), gen, 8)
    cells = eps = None
    if disorder:
        cells = _smooth((Ny - 1, Nx - 1), gen, 6) > -1.645  # about 5% of the area removed
        near = torch.zeros((Ny, Nx), dtype=torch.bool, device="cuda")
        for j in (0, 1):
            for i in (0, 1):
                near[j:Ny - 1 + j, i:Nx - 1 + i] |= cells
        psi = torch.where(near, psi, torch.zeros_like(psi))
        if pinned:
            eps = (1.0 + 0.2 * _smooth((Ny, Nx), gen)).to(real)
    return psi.to(torch.complex64 if dtype == "float32" else torch.complex128), a.to(real), b.to(real), cells, eps


def _host(t):
    """The (Nx, Ny) host array of a (Ny, Nx) device field."""
    return t.cpu().numpy().T


def _solver(Nx, Ny, kappa, disorder, dtype, seed, pinned):
    psi, a, b, cells, eps = _fields(Nx, Ny, kappa, disorder, dtype, seed, pinned)
    gl = GLSolver(Nx=Nx, Ny=Ny, dx=DX, dy=DX, dtype=np.float32 if dtype == "float32" else np.float64,
                  order_parameter=_host(psi), gl_parameter=kappa if kappa else np.inf, normal_conductivity=SIGMA,
                  homogeneous_external_field=H, material_tiling=None if cells is None else _host(cells),
                  linear_coefficient=1.0 if eps is None else _host(eps))
    gl.vars.vector_potential = (_host(a), _host(b))
    return gl


def _sizes(case):
    """The sides of a batch's instances: the largest sides over 1, 2, 4, 8, 16 (at least 33 nodes)."""
    if case["kind"] == "batch_cg":
        return [(case["Nx"], case["Ny"])] * case["count"]
    rng = np.random.default_rng(case["count"])  # the mix of sizes belongs to the case, not to the seed
    pick = lambda n: max(33, (n - 1) // int(rng.choice([1, 2, 4, 8, 16])) + 1)  # noqa: E731
    return [(pick(case["Nx"]), pick(case["Ny"])) for _ in range(case["count"])]


def _instance_kappa(case, k):
    """Batched time evolution mixes kappa, every third instance in the kappa = inf limit;
    a batched minimisation takes one of the two kinds."""
    if case["kind"] == "batch_td" and case["kappa"] and k % 3 == 2:
        return 0.0
    return case["kappa"]


def _pinned(case):
    """Pinning maps where the solvers take them into account throughout (the single-instance
    line search reads the scalar epsilon alone)."""
    return case["kind"] != "cg"


class _Handle:
    """A device array of the framework for torch (the CUDA array interface)."""

    def __init__(self, dev):
        self.dev = dev
        kind = {"f": "<f", "c": "<c"}[dev.dtype.kind] + str(dev.dtype.itemsize)
        self.__cuda_array_interface__ = {"shape": (dev.size,), "typestr": kind, "data": (dev.ptr, False),
                                         "version": 2, "strides": None}


def _tensor(dev):
    return torch.as_tensor(_Handle(dev), device="cuda")


class _State:
    def __init__(self, case, seed):
        self.kind, self.steps = case["kind"], case["steps"]
        if self.kind in ("batch_td", "batch_cg"):
            self.sims = [_solver(Nx, Ny, _instance_kappa(case, k), case["disorder"], case["dtype"], seed * 1000 + k,
                                 _pinned(case)) for k, (Nx, Ny) in enumerate(_sizes(case))]
            self.batch = (BatchTD if self.kind == "batch_td" else BatchCG)(self.sims)
        else:
            self.sims = [_solver(case["Nx"], case["Ny"], case["kappa"], case["disorder"], case["dtype"], seed,
                                 _pinned(case))]
        self.start = [(gl.vars.order_parameter_h().copy(), gl.vars.vector_potential_h().copy()) for gl in self.sims]

    def restore(self):
        for gl, (psi, ab) in zip(self.sims, self.start):
            gl.vars.order_parameter_h().copy_from(psi)
            if gl.params.solveA:
                gl.vars.vector_potential_h().copy_from(ab)


def prepare(case, seed):
    return _State(case, seed)


def run(s):
    gl = s.sims[0]
    if s.kind == "analysis":
        gl.solve.vortices_detected = False  # as every solver call leaves it
        B, (Jx, Jy), (Sx, Sy) = gl.observables.bulk_observables()
        found = gl.vortex_detector.vortices
        table = np.zeros((3, B.size // 16 + 16), dtype=found[0].dtype)  # x, y, v, one shape for any number of vortices
        n = min(len(found[0]), table.shape[1])
        for row, values in zip(table, found):
            row[:n] = values[:n]
        return {"F": gl.observables.free_energy, "B": B, "Jx": Jx, "Jy": Jy, "Sx": Sx, "Sy": Sy, "vortices": table}
    if s.kind == "batch_cg":
        torch.cuda.synchronize()  # torch may still be gathering the last results from the buffers written next
    s.restore()
    if s.kind == "td":
        gl.solve.td(dt=DT, Nt=s.steps)
        out = {"psi": _tensor(gl.vars.order_parameter_h())}
        if gl.params.solveA:
            out["ab"] = _tensor(gl.vars.vector_potential_h())
        return out
    if s.kind == "cg":
        gl.solve.cg(n_iter=s.steps)
        out = {"psi": _tensor(gl.vars.order_parameter_h()), "F": gl.observables.free_energy}
        if gl.params.solveA:
            out["ab"] = _tensor(gl.vars.vector_potential_h())
        return out
    if s.kind == "batch_td":
        s.batch.td(dt=DT, Nt=s.steps)
        return {"psi": [_tensor(g.vars.order_parameter_h()) for g in s.sims],
                "ab": [_tensor(g.vars.vector_potential_h()) for g in s.sims if g.params.solveA]}
    s.batch.cg(max_iter=s.steps, rtol=1e-8)
    out = {"psi": torch.cat([_tensor(g.vars.order_parameter_h()) for g in s.sims])}
    if gl.params.solveA:
        out["ab"] = torch.cat([_tensor(g.vars.vector_potential_h()) for g in s.sims])
    return out


def work(case):
    """Each field read once and each result written once; operations of the sweeps and
    iterations that the stop rules ask for (about 12 psi sweeps and 3 A sweeps a step)."""
    s = 4 if case["dtype"] == "float32" else 8
    kind, steps = case["kind"], case["steps"]
    sizes = _sizes(case) if kind.startswith("batch") else [(case["Nx"], case["Ny"])]
    nbytes = flops = 0.0
    for k, (Nx, Ny) in enumerate(sizes):
        N, withA = Nx * Ny, bool(_instance_kappa(case, k))
        fields = 2 * s + 2 * s + (1 if case["disorder"] else 0) + (s if case["disorder"] and _pinned(case) else 0)
        if kind == "analysis":
            nbytes += N * (fields + s + 2 * s + 2 * s)
            flops += N * 150.0
            continue
        nbytes += N * (fields + 2 * s + (2 * s if withA else 0))
        if kind.endswith("td"):
            flops += N * steps * (12 * 40.0 + (3 * 36.0 + 40.0 if withA else 0.0))
        else:
            flops += N * steps * (450.0 if withA else 200.0)
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------- the same in 64 bits, plainly

def exact(case, seed):
    kind = case["kind"]
    if kind == "analysis":
        m = _Model(case, case["Nx"], case["Ny"], case["kappa"], seed)
        B, Jx, Jy, Sx, Sy = m.observables()
        return {"F": float(m.energy(m.psi, m.a, m.b)), "B": B.T, "Jx": Jx.T, "Jy": Jy.T, "Sx": Sx.T, "Sy": Sy.T,
                "vortices": None}
    if kind in ("td", "cg"):
        m = _Model(case, case["Nx"], case["Ny"], case["kappa"], seed)
        m.td(case["steps"]) if kind == "td" else m.cg(case["steps"], batch=False)
        out = {"psi": m.flat_psi()}
        if kind == "cg":
            out["F"] = float(m.energy(m.psi, m.a, m.b))
        if case["kappa"]:
            out["ab"] = m.flat_ab()
        return out
    psi, ab = [], []
    for k, (Nx, Ny) in enumerate(_sizes(case)):
        m = _Model(case, Nx, Ny, _instance_kappa(case, k), seed * 1000 + k)
        if kind == "batch_cg":
            m.cg(case["steps"], batch=True)
        else:
            m.td(case["steps"])
        psi.append(m.flat_psi())
        if _instance_kappa(case, k):
            ab.append(m.flat_ab())
    if kind == "batch_td":
        return {"psi": psi, "ab": ab}
    return {"psi": torch.cat(psi), "ab": torch.cat(ab)} if ab else {"psi": torch.cat(psi)}


class _Model:
    """The lattice Ginzburg-Landau equations written out on (Ny, Nx) float64 tensors."""

    def __init__(self, case, Nx, Ny, kappa, seed):
        psi, a, b, cells, eps = _fields(Nx, Ny, kappa, case["disorder"], case["dtype"], seed, _pinned(case))
        rnd = (lambda v: float(np.float32(v))) if case["dtype"] == "float32" else float
        self.psi, self.a, self.b = psi.to(torch.complex128), a.double(), b.double()
        self.eps = torch.ones((), dtype=torch.float64, device="cuda") if eps is None else eps.double()
        self.k2, self.rho, self.H, self.dt = rnd(kappa) ** 2, rnd(1.0 / SIGMA), rnd(H), rnd(DT)
        self.stop = rnd(STOP)
        self.kappa = kappa
        full = torch.zeros((Ny + 1, Nx + 1), dtype=torch.float64, device="cuda")
        full[1:Ny, 1:Nx] = 1.0 if cells is None else cells.double()
        mm, mp, pm, pp = full[:-1, :-1], full[1:, :-1], full[:-1, 1:], full[1:, 1:]
        self.on_a = torch.maximum(pm, pp)[:, :-1]     # a(i, j) touches the material
        self.on_b = torch.maximum(mp, pp)[:-1, :]
        self.w_a = 0.5 * (pm + pp)[:, :-1]            # link weights of the free energy
        self.w_b = 0.5 * (mp + pp)[:-1, :]
        self.w_n = 0.25 * (mm + mp + pm + pp)
        self.inside = torch.maximum(torch.maximum(mm, mp), torch.maximum(pm, pp))
        self.links = (torch.maximum(mm, mp) + torch.maximum(pm, pp) + torch.maximum(mm, pm)
                      + torch.maximum(mp, pp)) / DX ** 2

    def flat_psi(self):
        return self.psi.reshape(-1)

    def flat_ab(self):
        return torch.cat([self.a.reshape(-1), self.b.reshape(-1)])

    @staticmethod
    def _met(r, stop):
        return int(min(1e4 * r / stop, 1e8)) < 10000

    @staticmethod
    def _ua(a):
        return torch.polar(torch.ones_like(a), -DX * a)

    # -- time evolution: backward Euler, Jacobi sweeps to the stop rule
    def td(self, steps):
        for _ in range(steps):
            self._psi_step()
            if self.kappa:
                self._a_step()

    def _psi_step(self):
        c = self.dt / DX ** 2
        ua, ub = self._ua(self.a) * (c * self.on_a), self._ua(self.b) * (c * self.on_b)
        rhs = self.psi
        den = 1.0 + self.dt * (rhs.real ** 2 + rhs.imag ** 2 - self.eps + self.links)
        keep = self.inside / den
        p = rhs
        for _ in range(1024):
            q = rhs.clone()
            q[:, :-1] += ua * p[:, 1:]
            q[:, 1:] += ua.conj() * p[:, :-1]
            q[:-1] += ub * p[1:]
            q[1:] += ub.conj() * p[:-1]
            q *= keep
            d = torch.view_as_real(q - p).abs().max().item()
            p = q
            if self._met(d, self.stop):
                break
        self.psi = p

    def _currents(self, psi, a, b):
        ja = (psi[:, :-1].conj() * self._ua(a) * psi[:, 1:]).imag / DX
        jb = (psi[:-1].conj() * self._ua(b) * psi[1:]).imag / DX
        return ja, jb

    def _curls(self, a, b, H_edge):
        """Sums over the other links of the two cells at a link (curl curl A without its
        diagonal, doubled at the sample's edge, where the field is H_edge outside)."""
        h2 = 1.0 / DX ** 2
        ta, tb = torch.zeros_like(a), torch.zeros_like(b)
        db = (b[:, 1:] - b[:, :-1]) * h2
        ta[1:] += h2 * a[:-1] + db
        ta[:-1] += h2 * a[1:] - db
        da = (a[1:] - a[:-1]) * h2
        tb[:, 1:] += h2 * b[:, :-1] + da
        tb[:, :-1] += h2 * b[:, 1:] - da
        ta[0] *= 2.0
        ta[-1] *= 2.0
        tb[:, 0] *= 2.0
        tb[:, -1] *= 2.0
        s = 2.0 * H_edge / DX
        ta[0] += s
        ta[-1] -= s
        tb[:, 0] -= s
        tb[:, -1] += s
        return ta, tb

    def _a_step(self):
        dr, drk = self.dt * self.rho, self.dt * self.rho * self.k2
        den = 1.0 + 2.0 * drk / DX ** 2
        a0, b0 = self.a, self.b
        before, cur = None, (a0, b0)
        for j in range(1024):
            # the supercurrent of an odd sweep is that of the sweep before it
            sa, sb = cur if j % 2 == 0 else before
            if j % 2 == 0:
                ja, jb = self._currents(self.psi, sa, sb)
                ja, jb = ja * self.on_a, jb * self.on_b
            ta, tb = self._curls(cur[0], cur[1], self.H)
            new = ((a0 + dr * ja + drk * ta) / den, (b0 + dr * jb + drk * tb) / den)
            d = max((new[0] - cur[0]).abs().max().item(), (new[1] - cur[1]).abs().max().item())
            before, cur = cur, new
            if self._met(d, self.stop):
                break
        self.a, self.b = cur

    # -- free energy, currents and field
    def _grads(self, psi, a, b):
        return psi[:, 1:] * self._ua(a) - psi[:, :-1], psi[1:] * self._ua(b) - psi[:-1]

    def _field(self, a, b):
        return (b[:, 1:] - b[:, :-1] - a[1:] + a[:-1]) / DX

    def _matter(self, psi, a, b, eps):
        p2 = psi.real ** 2 + psi.imag ** 2
        ga, gb = self._grads(psi, a, b)
        e = (self.w_n * (0.5 * p2 - eps) * p2).sum()
        e = e + (self.w_a * (ga.real ** 2 + ga.imag ** 2)).sum() / DX ** 2
        return DX ** 2 * (e + (self.w_b * (gb.real ** 2 + gb.imag ** 2)).sum() / DX ** 2)

    def _magnetic(self, a, b):
        return DX ** 2 * self.k2 * (self._field(a, b) - self.H).square().sum()

    def energy(self, psi, a, b):
        f = self._matter(psi, a, b, self.eps)
        return f + self._magnetic(a, b) if self.kappa else f

    def observables(self):
        ja, jb = self._currents(self.psi, self.a, self.b)
        ja, jb = ja * self.w_a, jb * self.w_b
        if not self.kappa:
            return self._field(self.a, self.b), ja, jb, ja, jb
        ta, tb = self._curls(self.a, self.b, self.H)
        h2 = 1.0 / DX ** 2
        return (self._field(self.a, self.b), self.k2 * (2.0 * h2 * self.a - ta), self.k2 * (2.0 * h2 * self.b - tb),
                ja, jb)

    # -- conjugate gradients (Polak-Ribiere, minimum of the line polynomial)
    def _gradient(self, batch):
        psi, a, b = (t.detach().requires_grad_(True) for t in (self.psi, self.a, self.b))
        self._matter(psi, a, b, self.eps).backward()
        g = [psi.grad, a.grad, b.grad]
        if not self.kappa:
            return g[:1]
        a2, b2 = (t.detach().requires_grad_(True) for t in (self.a, self.b))
        self._magnetic(a2, b2).backward()
        if not batch:  # the single-instance form counts the field outside the edge as well
            for t in (a2.grad[0], a2.grad[-1], b2.grad[:, 0], b2.grad[:, -1]):
                t *= 2.0
        return [g[0], g[1] + a2.grad, g[2] + b2.grad]

    def _poly(self, d):
        """c[i, k]: coefficient of (psi step)^i (A step)^k, phases expanded to fourth order."""
        P, D, eps = self.psi, d[0], self.eps
        c = np.zeros((5, 5))
        p2, d2 = P.real ** 2 + P.imag ** 2, D.real ** 2 + D.imag ** 2
        tw = 2.0 * (P.real * D.real + P.imag * D.imag)
        w = self.w_n
        c[0, 0] = (w * (0.5 * p2 - eps) * p2).sum()
        c[1, 0] = (w * tw * (p2 - eps)).sum()
        c[2, 0] = (w * (p2 * d2 + 0.5 * tw * tw - eps * d2)).sum()
        c[3, 0] = (w * tw * d2).sum()
        c[4, 0] = (w * 0.5 * d2 * d2).sum()
        top = 0.0
        for ax, A, wl in ((1, self.a, self.w_a), (0, self.b, self.w_b)):
            n = P.shape[ax]
            P0, P1, D0, D1 = P.narrow(ax, 0, n - 1), P.narrow(ax, 1, n - 1), D.narrow(ax, 0, n - 1), D.narrow(ax, 1, n - 1)
            u, wl = self._ua(A), wl / DX ** 2
            gp, gd = P1 * u - P0, D1 * u - D0
            c[0, 0] += (wl * gp.abs() ** 2).sum()
            c[1, 0] += 2.0 * (wl * (gp.conj() * gd).real).sum()
            c[2, 0] += (wl * gd.abs() ** 2).sum()
            if not self.kappa:
                continue
            ph = DX * d[1 if ax == 1 else 2]
            top = max(top, ph.abs().max().item())
            for i, z in enumerate((P0 * (P1 * u).conj(), P0 * (D1 * u).conj() + D0 * (P1 * u).conj(),
                                   D0 * (D1 * u).conj())):
                c[i, 1] += 2.0 * (wl * z.imag * ph).sum()
                c[i, 2] += (wl * z.real * ph ** 2).sum()
                c[i, 3] -= (wl * z.imag * ph ** 3).sum() / 3.0
                c[i, 4] -= (wl * z.real * ph ** 4).sum() / 12.0
        if self.kappa:
            f, df = self._field(self.a, self.b) - self.H, self._field(d[1], d[2])
            c[0, 0] += self.k2 * f.square().sum()
            c[0, 1] += 2.0 * self.k2 * (f * df).sum()
            c[0, 2] += self.k2 * df.square().sum()
        return c * DX ** 2, top

    @staticmethod
    def _minimum(c, top):
        """The minimum of the line polynomial reached from (0, 0) by damped Newton steps,
        with no link phase moved by more than half a radian."""
        pv, pd = np.polynomial.polynomial.polyval2d, np.polynomial.polynomial.polyder
        cx, cy = pd(c, axis=0), pd(c, axis=1)
        cxx, cxy, cyy = pd(cx, axis=0), pd(cx, axis=1), pd(cy, axis=1)
        most = 0.5 / top if top > 0.0 else 0.0
        x = y = 0.0
        for _ in range(80):
            gx, gy = pv(x, y, cx), pv(x, y, cy)
            hxx, hxy, hyy = pv(x, y, cxx), pv(x, y, cxy), pv(x, y, cyy)
            if top == 0.0:
                gy, hxy, hyy = 0.0, 0.0, 1.0
            det = hxx * hyy - hxy * hxy
            dx, dy = -gx, -gy
            if hxx > 0.0 and det > 0.0:
                dx, dy = -(hyy * gx - hxy * gy) / det, -(hxx * gy - hxy * gx) / det
            f, t = pv(x, y, c), 1.0
            for _ in range(60):
                sx, sy = t * dx, min(max(y + t * dy, -most), most) - y
                if pv(x + sx, y + sy, c) < f:
                    break
                t *= 0.5
            else:
                break
            x, y = x + sx, y + sy
            if abs(sx) + abs(sy) <= 1e-15 * (abs(x) + abs(y)):
                break
        return x, y

    def cg(self, steps, batch):
        g, old, last = self._gradient(batch), None, None
        for it in range(steps):
            if it == 0:
                d = [-t for t in g]
            else:
                dot = lambda u, v: (u.conj() * v).real.sum().item() if u.is_complex() else (u * v).sum().item()  # noqa: E731
                beta = max(dot(g[0], g[0] - old[0]) / dot(old[0], old[0]), 0.0)
                betas = [beta]
                if self.kappa:
                    num = dot(g[1], g[1] - old[1]) + dot(g[2], g[2] - old[2])
                    beta = max(num / (dot(old[1], old[1]) + dot(old[2], old[2])), 0.0)
                    betas += [beta, beta]
                d = [q * u - t for q, u, t in zip(betas, d, g)]
            x, y = self._minimum(*self._poly(d))
            self.psi = self.psi + x * d[0]
            if self.kappa:
                self.a, self.b = self.a + y * d[1], self.b + y * d[2]
            if not batch:
                f = float(self.energy(self.psi, self.a, self.b))
                if last is not None and abs(f / last - 1.0) < 1e-6:
                    break
                last = f
            old, g = g, self._gradient(batch)
