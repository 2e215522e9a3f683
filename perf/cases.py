"""The calls whose speed is measured: whole runs of the fused state, steps of
the per-function integrator, one right-hand side of it, and gradients through
the adjoint, over the sizes the framework's own configurations use.

A case is a dict of plain values:

  kind       "fused" (FusedState: load, evolve, store), "step" (core.Integrator
             advancing a saved state), "rhs" (the four per-function calls of one
             right-hand side) or "grad" (adjoint.FlavorObjective, forward and
             backward)
  nf         2 or 3 flavours
  nx, ny, nz periodic cells; a dimension of one cell has a one-cell stencil
  ndir       momentum directions per cell (one particle each)
  order      shape factor order, 0 to 2
  precision  "fp64" or "fp32" (FP32-bulk; per-function calls are FP64 only)
  steps      RK4 steps of one pass
  shuffled   particles in a random order instead of the initializer's

``prepare`` makes the state of a run under way: every direction's particles
form the initial lattice of cell centres, shifted along the direction by the
distance travelled so far (all particles move at c), with pure flavour states
near the electron flavour and a forward-peaked nubar distribution.  ``exact``
evaluates the same pass in plain float64 torch.

FP32-bulk results are returned as float32, which holds them without loss:
that is what the state keeps.  Positions are float64 in both precisions.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from emu_amd import adjoint, core
from emu_amd.params import TestParams

# physical constants, cgs
EV = 1.60218e-12
C = 2.99792458e10
HBAR = 1.05457266e-27
GF = 1.1663787e-5 / (1e9 * 1e9 * EV * EV) * (HBAR * C) ** 3

NDENS = 4.89e32     # nu and nubar number density, cm^-3
FLUXFACBAR = 0.33   # nubar flux factor along +z
ENERGY = 50e6 * EV
CFL = 0.4
MASS_EV = {2: (-math.sqrt(7.4e-5), 0.0, 0.0), 3: (0.0, math.sqrt(7.4e-5), math.sqrt(2.5e-3))}
ANGLES = {2: (33.82, 0.0, 0.0), 3: (33.82, 48.3, 222.0)}  # theta12, theta13, deltaCP in degrees
DX = 0.5            # cell edge, cm


def _case(name, kind, nf, n, ndir, precision="fp64", steps=1, order=2, shuffled=False):
    c = dict(kind=kind, nf=nf, nx=n[0], ny=n[1], nz=n[2], ndir=ndir, order=order, precision=precision, steps=steps,
             shuffled=shuffled)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the headline workload, a 3-flavour fast-flavour box: a production run's
        # time between two outputs, in each precision
        _case("fused_fp32_64cube", "fused", 3, (64, 64, 64), 92, "fp32", steps=6),
        _case("fused_fp64_64cube", "fused", 3, (64, 64, 64), 92, "fp64", steps=4),
        # the 1-D fiducial run: few cells with many directions each
        _case("fused_fp32_1d", "fused", 3, (1, 1, 1024), 378, "fp32", steps=60),
        # a workstation-sized 2-flavour box with few directions per cell
        _case("fused_fp64_16cube", "fused", 2, (16, 16, 16), 26, "fp64", steps=50),
        # a mid-sized 2-flavour box
        _case("fused_fp32_32cube", "fused", 2, (32, 32, 32), 92, "fp32", steps=15),
        # the smallest run: one homogeneous cell, as the MSW and bipolar decks
        _case("fused_fp64_onecell", "fused", 2, (1, 1, 1), 24, "fp64", steps=100),
        # a domain and a direction set that divide by nothing
        _case("fused_fp64_ragged", "fused", 3, (37, 29, 23), 127, "fp64", steps=8),
        # the drop-in integrator on the per-function calls
        _case("step_32cube", "step", 3, (32, 32, 32), 92),
        _case("step_16cube", "step", 2, (16, 16, 16), 26),
        # one right-hand side from a caller with its own integrator, its
        # particles in no particular order
        _case("rhs_shuffled", "rhs", 3, (35, 28, 31), 61, shuffled=True),
        # gradients of the final flavour coherence: the 2-flavour adjoint box,
        # and a 3-flavour FP32-bulk one
        _case("grad_fp64_32cube", "grad", 2, (32, 32, 32), 92, "fp64", steps=4),
        _case("grad_fp32_nf3", "grad", 3, (24, 20, 16), 92, "fp32", steps=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any kind, 1-D to 3-D, 10^2 to 10^7 particles."""
    kind = rng.choice(("fused", "fused", "fused", "step", "rhs", "grad"))
    nf = rng.choice((2, 3))
    precision = rng.choice(("fp64", "fp32")) if kind in ("fused", "grad") else "fp64"
    ndir = _log_int(rng, 12, 400)
    most = {"fused": 10e6, "step": 3e6, "rhs": 3e6, "grad": 2e6}[kind]
    cells = _log_int(rng, 8, most / ndir)
    if rng.random() < 0.25:
        n = (1, 1, max(4, min(cells, 2048)))
    else:
        edge = cells ** (1.0 / 3.0)
        n = tuple(max(3, int(round(edge * rng.uniform(0.75, 1.3)))) for _ in range(3))
    np_ = n[0] * n[1] * n[2] * ndir
    steps = {"fused": rng.randint(3, max(4, min(20, int(9e7 / np_)))), "step": 1, "rhs": 1,
             "grad": rng.randint(2, 5)}[kind]
    order = rng.choice((1, 2, 2, 2))
    return _case(None, kind, nf, n, ndir, precision, steps, order, rng.random() < 0.25 and kind != "grad")


# ---- inputs -----------------------------------------------------------------

def _lengths(case):
    """Domain edges: cells of DX along dimensions the case resolves, 1 cm along others."""
    return [DX * n if n > 1 else 1.0 for n in (case["nx"], case["ny"], case["nz"])]


def _params(case) -> TestParams:
    m, a, L = MASS_EV[case["nf"]], ANGLES[case["nf"]], _lengths(case)
    return TestParams.from_dict(dict(
        nf=case["nf"], shape_order=case["order"], ncell=(case["nx"], case["ny"], case["nz"]), Lx=L[0], Ly=L[1],
        Lz=L[2], mass1_eV=m[0], mass2_eV=m[1], mass3_eV=m[2], theta12_degrees=a[0], theta13_degrees=a[1],
        deltaCP_degrees=a[2], cfl_factor=CFL, flavor_cfl_factor=CFL, maxError=1e-6, rho_g_ccm=0.0, Ye=1.0))


def _herm(nf):
    """(i, j, is_imaginary) of each Hermitian component."""
    out = []
    for i in range(nf):
        for j in range(i, nf):
            out.append((i, j, False))
            if j > i:
                out.append((i, j, True))
    return out


def _su_length(f, nf):
    """|f|_SU of component rows f[nh]."""
    comp = _herm(nf)
    s = sum(f[c] ** 2 for c, (i, j, _) in enumerate(comp) if i != j)
    diag = [f[c] for c, (i, j, _) in enumerate(comp) if i == j]
    for l in range(1, nf):
        bc = (sum(diag[:l]) - l * diag[l]) * math.sqrt(2.0 / (l * (l + 1)))
        s = s + (bc / 2) ** 2
    return s.sqrt()


def _pure_state(nf, np_, g, dev):
    """Component rows of |psi><psi|, psi near the electron flavour."""
    psi = [torch.ones(np_, dtype=torch.complex128, device=dev)]
    for _ in range(nf - 1):
        e = torch.randn(2, np_, dtype=torch.float64, device=dev, generator=g)
        psi.append(0.02 * torch.complex(e[0], e[1]))
    norm = sum(p.abs() ** 2 for p in psi).sqrt()
    rows = []
    for i, j, im in _herm(nf):
        m = (psi[i] / norm) * (psi[j] / norm).conj()
        rows.append(m.imag if im else m.real)
    return torch.stack(rows)


def _particles(case, seed):
    """Positions [3][np], attributes by name and ids of the case's particles."""
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    nf, nd, n, L = case["nf"], case["ndir"], (case["nx"], case["ny"], case["nz"]), _lengths(case)
    k = torch.arange(nd, dtype=torch.float64, device=dev)
    uz = 1.0 - (2.0 * k + 1.0) / nd                        # Fibonacci sphere
    r, phi = (1.0 - uz * uz).sqrt(), math.pi * (3.0 - math.sqrt(5.0)) * k
    u = torch.stack([r * phi.cos(), r * phi.sin(), uz])
    cells = n[0] * n[1] * n[2]
    np_ = cells * nd
    # cells with z fastest, then directions
    cell = torch.arange(cells, device=dev)
    ijk = (cell // (n[1] * n[2]), (cell // n[2]) % n[1], cell % n[2])
    travelled = DX * (1.0 + 3.0 * torch.rand(1, dtype=torch.float64, device=dev, generator=g))
    pos = torch.empty(3, np_, dtype=torch.float64, device=dev)
    for d in range(3):
        centre = (ijk[d].double() + 0.5) * (L[d] / n[d])
        pos[d] = torch.remainder(centre[:, None] + u[d] * travelled, L[d]).reshape(-1)
    a = {"pup%s" % x: (u[d] * ENERGY).repeat(cells) for d, x in enumerate("xyz")}
    a["pupt"] = torch.full((np_,), ENERGY, dtype=torch.float64, device=dev)
    w = NDENS * (L[0] / n[0]) * (L[1] / n[1]) * (L[2] / n[2]) / nd
    a["N"] = torch.full((np_,), w, dtype=torch.float64, device=dev)
    a["Nbar"] = w * (1.0 + 3.0 * FLUXFACBAR * uz).repeat(cells)
    a["f"], a["fbar"] = _pure_state(nf, np_, g, dev), _pure_state(nf, np_, g, dev)
    a["L"], a["Lbar"] = _su_length(a["f"], nf), _su_length(a["fbar"], nf)
    ids = torch.arange(1, np_ + 1, dtype=torch.int64, device=dev)
    if case["shuffled"]:
        p = torch.randperm(np_, device=dev, generator=g)
        pos, ids = pos[:, p].contiguous(), ids[p]
        a = {key: v[..., p].contiguous() for key, v in a.items()}
    return pos, a, ids


def _container(emu, case, seed):
    pos, a, ids = _particles(case, seed)
    K, nh = emu.K, emu.nh
    c = core.FlavoredNeutrinoContainer(emu, pos.shape[1])
    c.pos.copy_(pos)
    c.rdata[K["x"]:K["z"] + 1].copy_(pos)
    for key in ("pupx", "pupy", "pupz", "pupt", "N", "Nbar", "L", "Lbar"):
        c.rdata[K[key]].copy_(a[key])
    c.rdata[K["f00_Re"]:K["f00_Re"] + nh].copy_(a["f"])
    c.rdata[K["f00_Rebar"]:K["f00_Rebar"] + nh].copy_(a["fbar"])
    c.ids.copy_(ids)
    return c


# ---- the measured calls -----------------------------------------------------

class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case = case
    s.emu = core.Emu(_params(case))
    s.parts = _container(s.emu, case, seed)
    kind = case["kind"]
    if kind == "fused":
        s.out = core.FlavoredNeutrinoContainer(s.emu, s.parts.np)
        s.st = core.FusedState(s.emu, s.parts.np, case["precision"])
    elif kind == "step":
        start = core.FlavoredNeutrinoContainer(s.emu, s.parts.np)
        start.copyParticles(s.parts)
        s.integrator = core.Integrator(s.emu, start)
        s.dt = s.integrator.dt
    elif kind == "rhs":
        s.grid = core.MultiFab(s.emu)
        s.grid.FillBoundary()
        s.F = core.FlavoredNeutrinoContainer(s.emu, s.parts.np)
    else:
        grid = core.MultiFab(s.emu)
        core.deposit_to_mesh(s.parts, grid)
        dt = core.compute_dt(grid, s.parts.Vvac_max())
        s.problem = adjoint.AdjointProblem(s.emu, s.parts, dt=dt, nsteps=case["steps"], precision=case["precision"])
        s.parts = None
    return s


def _attributes(emu, c, dtype=torch.float64):
    """A container's attributes by group."""
    K, nh, r = emu.K, emu.nh, c.rdata
    groups = {"time": r[K["time"]], "x": r[K["x"]:K["z"] + 1], "pup": r[K["pupx"]:K["pupt"] + 1], "N": r[K["N"]],
              "L": r[K["L"]], "f": r[K["f00_Re"]:K["f00_Re"] + nh], "Nbar": r[K["Nbar"]], "Lbar": r[K["Lbar"]],
              "fbar": r[K["f00_Rebar"]:K["f00_Rebar"] + nh]}
    return {k: v if k == "x" else v.to(dtype) for k, v in groups.items()}


def run(s):
    case, emu = s.case, s.emu
    kind = case["kind"]
    dtype = torch.float32 if case["precision"] == "fp32" else torch.float64
    if kind == "fused":
        s.st.load(s.parts)
        s.st.evolve(case["steps"])
        s.st.store(s.out)
        return {"pos": s.out.pos, "ids": s.out.ids, **_attributes(emu, s.out, dtype)}
    if kind == "step":
        it = s.integrator
        it.old.copyParticles(s.parts)
        it.dt, it.time = s.dt, 0.0
        for _ in range(case["steps"]):
            it.advance()
        return {"pos": it.old.pos, "ids": it.old.ids, "dt": it.dt, **_attributes(emu, it.old)}
    if kind == "rhs":
        core.deposit_to_mesh(s.parts, s.grid)
        s.grid.FillBoundary()
        s.F.copyParticles(s.parts)
        core.interpolate_rhs_from_mesh(s.F, s.grid)
        return {"grid": s.grid.data[3:], "pos": s.F.pos, **_attributes(emu, s.F)}
    f0 = s.problem.f0.clone().requires_grad_(True)
    ratio = torch.ones((), dtype=dtype, device=emu.device, requires_grad=True)
    loss = torch.log(adjoint.FlavorObjective.apply(f0, ratio, s.problem)).to(dtype)
    loss.backward()
    return {"loss": loss.detach(), "f0_grad": f0.grad, "ratio_grad": ratio.grad}


def work(case):
    """Compulsory bytes and operations of one pass.

    A fused step is the 3-register RK4 whose mesh coupling deposits before every
    gather: 65 + 20 S values per particle (S = 2 NF^2 flavour reals; 27 of them
    are float64 positions) and 12 grid passes of 4 NF^2 fields.  A step's 4
    deposits and 4 gathers take 27 x 4 NF^2 multiply-adds per particle each, and
    its commutators about 8 NF^3."""
    nf = case["nf"]
    nh, S = nf * nf, 2 * nf * nf
    cells = case["nx"] * case["ny"] * case["nz"]
    np_ = cells * case["ndir"]
    nt = 1
    for n in (case["nx"], case["ny"], case["nz"]):
        nt *= 3 if n > 1 else 1
    e = 4 if case["precision"] == "fp32" else 8
    step_bytes = np_ * (8 * 27 + e * (65 + 20 * S - 27)) + 12.0 * cells * 4 * nh * 8
    step_flops = np_ * 4.0 * (2 * 2 * nt * 4 * nh + 2 * 2 * 8 * nf ** 3)
    attrs = 3 + 12 + S
    if case["kind"] == "fused":
        # the load and the store: the caller's attributes in, the result out
        return {"bytes": case["steps"] * step_bytes + 2 * np_ * 8.0 * attrs, "flops": case["steps"] * step_flops}
    if case["kind"] == "step":
        return {"bytes": case["steps"] * step_bytes + 2 * np_ * 8.0 * attrs, "flops": case["steps"] * step_flops}
    if case["kind"] == "rhs":
        return {"bytes": np_ * 8.0 * (2 * attrs) + cells * 8.0 * nh * 8 * 2,
                "flops": np_ * (2.0 * nt * 8 * nh + 2.0 * nt * 4 * nh + 2 * 8 * nf ** 3)}
    # a gradient is the forward run and its replay, and a reverse step of twice a forward step's work
    return {"bytes": 4.0 * case["steps"] * step_bytes, "flops": 4.0 * case["steps"] * step_flops}


# ---- the same passes in plain float64 torch -----------------------------------

class _Model:
    """Deposit, gather and flavour right-hand side of particles grouped by cell.

    Flavour states are component rows [nh][np].  The sums over a cell's
    particles and over its 27 neighbours are batched matrix products on the
    particles padded to [cells][P] (padding has zero weights)."""

    def __init__(self, case, pos, pup, pupt):
        self.nf, self.nh = case["nf"], case["nf"] ** 2
        self.comp = _herm(self.nf)
        self.n = (case["nx"], case["ny"], case["nz"])
        self.L = _lengths(case)
        self.dx = [l / k for l, k in zip(self.L, self.n)]
        self.cells = self.n[0] * self.n[1] * self.n[2]
        self.volume = self.dx[0] * self.dx[1] * self.dx[2]
        self.order = [case["order"] if k > 1 else 0 for k in self.n]
        self.pupt, self.v = pupt, pup / pupt
        self.sign = torch.tensor([1.0 if im else -1.0 for _, _, im in self.comp], dtype=torch.float64,
                                 device=pos.device)
        m = [x * EV / C ** 2 for x in MASS_EV[self.nf]]
        t12, t13, dcp = (math.radians(x) for x in ANGLES[self.nf])
        c, sn = math.cos, math.sin
        U = np.array([[c(t12), sn(t12), 0], [-sn(t12), c(t12), 0], [0, 0, 1]], dtype=complex)
        if self.nf == 3:
            e = np.exp(-1j * dcp)
            U13 = np.array([[c(t13), 0, sn(t13) * e], [0, 1, 0], [-sn(t13) / e, 0, c(t13)]])
            U = np.array([[c(t13), 0, sn(t13)], [0, 1, 0], [-sn(t13), 0, c(t13)]]) @ U13 @ U
        M2 = (U @ np.diag([x * x for x in m]) @ U.conj().T)[:self.nf, :self.nf]
        self.vac = [(M2[i, j].imag if im else M2[i, j].real) * C ** 4 / (2 * HBAR) for i, j, im in self.comp]
        d = [x * x for x in m[:self.nf]]
        diag = torch.tensor([d[i] if i == j else 0.0 for i, j, _ in self.comp], dtype=torch.float64)
        self.vvac = float(_su_length(diag, self.nf)) * C ** 4 / ENERGY
        self.place(pos)

    def place(self, pos):
        """Bin the particles: their cells, stencil weights and padded lists."""
        idx, self.w = [], []
        for d in range(3):
            delta = pos[d] / self.dx[d]
            i = torch.floor(delta)
            o = delta - i - 0.5
            if self.order[d] == 2:
                w = (0.5 * (0.5 - o) ** 2, 0.75 - o * o, 0.5 * (0.5 + o) ** 2)
            elif self.order[d] == 1:
                w = ((-o).clamp(min=0), 1 - o.abs(), o.clamp(min=0))
            else:
                w = (torch.zeros_like(o), torch.ones_like(o), torch.zeros_like(o))
            idx.append(torch.remainder(i.long(), self.n[d]))
            self.w.append(w)
        self.idx = idx
        self.cell = (idx[2] * self.n[1] + idx[1]) * self.n[0] + idx[0]
        count = torch.bincount(self.cell, minlength=self.cells)
        order = torch.argsort(self.cell, stable=True)
        within = torch.empty_like(order)
        start = torch.cumsum(count, 0) - count
        within[order] = torch.arange(order.numel(), device=order.device) - start[self.cell[order]]
        self.P = max(1, int(count.max()))
        self.slot = self.cell * self.P + within
        wx, wy, wz = self.w
        stencil = torch.stack([wx[i] * wy[j] * wz[k] for k in range(3) for j in range(3) for i in range(3)], 1)
        self.W = self._pad(stencil)

    def _pad(self, x):
        """Rows [np][q] to [cells][P][q]."""
        out = torch.zeros(self.cells * self.P, x.shape[1], dtype=x.dtype, device=x.device)
        return out.index_copy(0, self.slot, x).view(self.cells, self.P, -1)

    def _roll(self, grid, t, sign):
        shift = (sign * (t // 9 - 1), sign * ((t // 3) % 3 - 1), sign * (t % 3 - 1))
        return torch.roll(grid, shift, dims=(0, 1, 2))

    def deposit(self, q):
        """Sum of w q over the particles, q [np][k] -> [nz][ny][nx][k]."""
        D = torch.bmm(self.W.transpose(1, 2).contiguous(), self._pad(q))
        D = D.view(self.n[2], self.n[1], self.n[0], 27, -1)
        return sum(self._roll(D[:, :, :, t], t, 1) for t in range(27))

    def gather(self, grid):
        """Sum of w grid over each particle's stencil -> [np][k]."""
        G = torch.stack([self._roll(grid, t, -1) for t in range(27)], 3).view(self.cells, 27, -1)
        return torch.bmm(self.W, G).view(self.cells * self.P, -1)[self.slot]

    def sources(self, f, fb, N, Nb):
        """N f - conj(Nbar fbar), and that times each velocity: [np][4 nh]."""
        q = (N * f + self.sign[:, None] * Nb * fb).t()
        return torch.cat([q] + [q * self.v[d][:, None] for d in range(3)], 1)

    def commutator(self, H, f):
        """-i (H f - f H) on component rows."""
        nf, zero = self.nf, None

        def entry(X, i, j):
            a, b = min(i, j), max(i, j)
            re = X[self.comp.index((a, b, False))]
            if i == j:
                return re, zero
            im = X[self.comp.index((a, b, True))]
            return re, im if i < j else -im

        def mul(x, y):
            re = x[0] * y[0]
            im = 0.0
            if x[1] is not None and y[1] is not None:
                re = re - x[1] * y[1]
            if x[1] is not None:
                im = im + x[1] * y[0]
            if y[1] is not None:
                im = im + x[0] * y[1]
            return re, im

        out = []
        for i, j, im in self.comp:
            re_s = im_s = 0.0
            for k in range(nf):
                a, b = mul(entry(H, i, k), entry(f, k, j)), mul(entry(f, i, k), entry(H, k, j))
                re_s, im_s = re_s + a[0] - b[0], im_s + a[1] - b[1]
            out.append(-re_s if im else im_s)
        return torch.stack(out)

    def rhs(self, f, fb, N, Nb):
        """d(f, fbar)/dt."""
        g = self.gather(self.deposit(self.sources(f, fb, N, Nb))).view(-1, 4, self.nh)
        inside = g[:, 0] - sum(self.v[d][:, None] * g[:, d + 1] for d in range(3))
        hs = (math.sqrt(2.0) * GF / self.volume / HBAR) * inside.t()
        hv = torch.stack([c / self.pupt for c in self.vac])
        return self.commutator(hv + hs, f), self.commutator(self.sign[:, None] * (hs - hv), fb)

    def dt(self, f, fb, N, Nb):
        """compute_dt from the deposit of a state."""
        rows = [c for c, (i, j, _) in enumerate(self.comp) if i == j]
        q = torch.cat([N * f[rows], Nb * fb[rows]]).t()
        top = float(self.deposit(q).max()) * 2.0 * self.nf * math.sqrt(2.0) * GF / self.volume
        return min(min(self.dx) / C * CFL, HBAR / (top + self.vvac) * CFL)

    def step(self, f, fb, N, Nb, dt):
        """One RK4 step of the flavour state; also the next step's dt."""
        k1 = self.rhs(f, fb, N, Nb)
        k2 = self.rhs(f + dt / 2 * k1[0], fb + dt / 2 * k1[1], N, Nb)
        k3 = self.rhs(f + dt / 2 * k2[0], fb + dt / 2 * k2[1], N, Nb)
        y4 = f + dt * k3[0], fb + dt * k3[1]
        k4 = self.rhs(*y4, N, Nb)
        new = [y + dt / 6 * (a + 2 * b + 2 * c + d) for y, a, b, c, d in zip((f, fb), k1, k2, k3, k4)]
        return new[0], new[1], y4

    def moved(self, pos, dt):
        """Positions after dt, and the index (0..26) of each particle's cell move."""
        new = torch.stack([torch.remainder(pos[d] + dt * C * self.v[d], self.L[d]) for d in range(3)])
        e = torch.zeros_like(self.cell)
        for d in (2, 1, 0):
            to = torch.remainder(torch.floor(new[d] / self.dx[d]).long(), self.n[d])
            m = torch.remainder(to - self.idx[d], self.n[d])
            e = 3 * e + torch.where(m == 0, 1, torch.where(m == 1, 2, 0))
        return new, e


def exact(case, seed):
    pos, a, ids = _particles(case, seed)
    np_, kind = pos.shape[1], case["kind"]
    names = ("pupx", "pupy", "pupz")
    pup, pupt = torch.stack([a[k] for k in names]), a["pupt"]
    if case["precision"] == "fp32":  # the momenta as FP32-bulk holds them: they carry the positions
        pup, pupt = pup.float().double(), pupt.float().double()
    f, fb, N, Nb = a["f"], a["fbar"], a["N"], a["Nbar"]
    model = _Model(case, pos, pup, pupt)
    if kind == "rhs":
        k, kb = model.rhs(f, fb, N, Nb)
        q, qb = (N * f).t(), (Nb * fb).t()
        cols = []
        for d in range(4):
            s = 1.0 if d == 0 else model.v[d - 1][:, None]
            cols += [q * s, qb * s]
        grid = model.deposit(torch.cat(cols, 1)).permute(3, 0, 1, 2)
        for d, n in enumerate((case["nz"], case["ny"], case["nx"])):  # ghost cells: periodic images
            ng = 1 + (1 + (case["order"] if n > 1 else 0)) // 2
            at = torch.remainder(torch.arange(-ng, n + ng, device=pos.device), n)
            grid = grid.index_select(d + 1, at)
        zero = torch.zeros(np_, dtype=torch.float64, device=pos.device)
        return {"grid": grid, "pos": pos, "time": zero + 1, "x": model.v * C, "pup": torch.zeros_like(a["f"][:4]),
                "N": zero, "L": zero, "f": k, "Nbar": zero, "Lbar": zero, "fbar": kb}
    if kind == "grad":
        dt = model.dt(f, fb, N, Nb)
        y0 = torch.cat([f, fb]).requires_grad_(True)
        ratio = torch.ones((), dtype=torch.float64, device=pos.device, requires_grad=True)
        y, yb, nh = y0[:model.nh], y0[model.nh:], model.nh
        for _ in range(case["steps"]):
            y, yb, _ = model.step(y, yb, N, Nb * ratio, dt)
            pos, _ = model.moved(pos, dt)
            model.place(pos)
        c01 = [c for c, (i, j, _) in enumerate(model.comp) if (i, j) == (0, 1)]
        loss = torch.log((model.deposit((N * y[c01]).t()) ** 2).sum())
        loss.backward()
        return {"loss": loss.detach(), "f0_grad": y0.grad, "ratio_grad": ratio.grad}
    # the fused state keeps its particles sorted by cell; particles that arrive in
    # a cell are ordered by their move, then as they were
    keep = [N, a["L"], Nb, a["Lbar"], a["pupx"], a["pupy"], a["pupz"], pupt]

    def reorder(o):
        nonlocal pos, f, fb, ids, keep
        pos, f, fb, ids = pos[:, o], f[:, o], fb[:, o], ids[o]
        keep = [x[o] for x in keep]
        model.v, model.pupt = model.v[:, o], model.pupt[o]
        model.place(pos)

    if kind == "fused":
        reorder(torch.argsort(model.cell, stable=True))
    time, dt = 0.0, model.dt(f, fb, keep[0], keep[2])
    for _ in range(case["steps"]):
        f, fb, y4 = model.step(f, fb, keep[0], keep[2], dt)
        next_dt = model.dt(*y4, keep[0], keep[2])
        pos, e = model.moved(pos, dt)
        time, dt = time + dt, next_dt
        if kind == "fused":
            model.place(pos)
            reorder(torch.argsort(model.cell * 27 + e, stable=True))
        else:
            model.place(pos)
    out = {"pos": pos, "ids": None, "time": torch.full_like(pos[0], time), "x": pos,
           "pup": torch.stack(keep[4:]), "N": keep[0], "L": keep[1], "f": f, "Nbar": keep[2], "Lbar": keep[3],
           "fbar": fb}
    return dict(out, dt=dt) if kind == "step" else out
