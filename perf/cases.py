"""Performance cases: what users of this solver have it do.

Four kinds of work, each through the public entry points of rism3d.py:

  solve      RISM3D.run: potentials, steps of the fixed-point loop, the
             thermodynamics (and g of every site where the case asks for
             fields, as the 'g' output letter does)
  batch      run_batch on many small solutes at once
  analysis   RISM3D.analysis on a state already solved: the forces on the
             solute's atoms and the per-atom energies (output letters d, b)
  transform  fft_noalloc on device buffers, forwards and there and back

The fixed-point loop runs for a set number of steps, as maxstep of an .inp
file sets it.  A converged solve takes 150 to 650 steps and stops within
tolerance of the fixed point rather than at a reproducible number, and its
per-step cost is the same; the step counts here stay where the iterates of
two builds that differ in rounding still agree closely.

Grids have 0.5 A spacing, the spacing of the benchmark workloads.  Solutes
are the seeded generators of gen_inputs.py, solvents the chi_vv files under
tests/golden.
"""
import functools
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "3d-rism-cuda-mpi_amd")
GOLDEN = os.path.join(ROOT, "tests", "golden")
SPACING = 0.5


@functools.lru_cache(maxsize=None)
def _package(name):
    """A module of the package, whose folder's name is no Python name."""
    if name in sys.modules:
        return sys.modules[name]
    spec = importlib.util.spec_from_file_location(name, os.path.join(PKG, name + ".py"))
    mod = importlib.util.module_from_spec(spec)
    sys.modules[name] = mod
    spec.loader.exec_module(mod)
    return mod


@functools.lru_cache(maxsize=None)
def _solvent(xvk):
    return _package("rism3d").read_xvk(os.path.join(GOLDEN, xvk + ".xvk"))


WATER = "tip3p_drism"           # 2 sites
SALT = "tip3p_nacl02_drism"     # 4 sites
KCL = "tip3p_kcl01_drism"       # 4 sites


def _solve(name, grid, solvent, atoms, steps, closure="KH", charge=0.0, anderson_m=0,
           precision=0, mixed_switch=0.0, mixed_block=0, fields=False):
    c = {"kind": "solve", "nx": grid[0], "ny": grid[1], "nz": grid[2], "solvent": solvent,
         "atoms": atoms, "steps": steps, "closure": closure, "charge": charge,
         "anderson_m": anderson_m, "precision": precision, "mixed_switch": mixed_switch,
         "mixed_block": mixed_block, "fields": fields}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one small molecule in the smallest box in use: launches and latency
        _solve("solve_48_small", (48, 48, 48), WATER, 8, 48),
        # the 64^3 / 24-atom benchmark molecule, with its distribution
        # functions brought back to the host
        _solve("solve_64_fields", (64, 64, 64), WATER, 24, 48, fields=True),
        # a box fitted to a long molecule: three different sides (so chi_vv
        # comes from the spline, not the cubic shell table), PSE-3, uncharged
        _solve("solve_ragged_pse3", (72, 90, 60), WATER, 30, 24, closure="PSE3"),
        # screening of small molecules: random-walk solutes of 8-60 atoms in
        # boxes fitted to each, solved as one batch
        {"name": "batch_small", "kind": "batch", "solutes": 48, "solvent": WATER, "steps": 48},
        # a peptide-sized cluster in salt water, non-cubic
        _solve("solve_144_salt", (144, 160, 128), SALT, 700, 48),
        # the benchmark configurations' other accelerator, Anderson(10)
        _solve("anderson10_160", (160, 160, 160), SALT, 400, 32, anderson_m=10),
        # a protein domain in salt water at 128 A
        _solve("solve_256_protein", (256, 256, 256), KCL, 1500, 40),
        # the headline grid, 512^3 at 256 A (a smaller protein than the
        # benchmark's, so that a pass stays short)
        _solve("solve_512_protein", (512, 512, 512), SALT, 1500, 32, charge=2.0),
        # the mixed-precision solve: its FP32 phase
        _solve("mixed_256", (256, 256, 256), WATER, 300, 8, precision=1),
        # forces on and energies of a small molecule's atoms
        {"name": "analysis_80", "kind": "analysis", "nx": 80, "ny": 72, "nz": 96,
         "solvent": WATER, "atoms": 40, "steps": 8, "closure": "KH"},
        # the transform by itself, a small uneven grid and a large one
        {"name": "transform_96_uneven", "kind": "transform", "nx": 96, "ny": 80, "nz": 60},
        {"name": "transform_256", "kind": "transform", "nx": 256, "ny": 256, "nz": 256},
    ]


# sizes that nx, ny and nz can all take (nz/2 is a transform length too)
SIZES = (32, 40, 48, 60, 64, 72, 80, 96, 128, 144, 160, 180, 192, 256)


def _sizes(rng, lo, hi):
    """Three grid sizes near one another, their scale spread over log size."""
    base = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    if rng.random() < 0.3:
        n = min(SIZES, key=lambda s: abs(math.log(s / base)))
        return (n, n, n)
    out = []
    for _ in range(3):
        want = base * math.exp(rng.uniform(-0.25, 0.25))
        out.append(min(SIZES, key=lambda s: abs(math.log(s / want))))
    return tuple(out)


def draw(rng):
    kind = rng.choice(["solve"] * 6 + ["batch", "analysis", "transform", "transform"])
    if kind == "batch":
        return {"kind": "batch", "solutes": rng.randint(6, 64), "solvent": WATER,
                "steps": rng.randint(24, 48)}
    if kind == "transform":
        nx, ny, nz = _sizes(rng, 32, 288)
        return {"kind": "transform", "nx": nx, "ny": ny, "nz": nz}
    if kind == "analysis":
        nx, ny, nz = _sizes(rng, 48, 110)
        return {"kind": "analysis", "nx": nx, "ny": ny, "nz": nz,
                "solvent": rng.choice([WATER, SALT]), "atoms": rng.randint(6, 120),
                "steps": rng.randint(4, 10), "closure": rng.choice(["KH", "KH", "PSE3"])}
    grid = _sizes(rng, 40, 280)
    n = grid[0] * grid[1] * grid[2]
    how = rng.choice(["an2"] * 4 + ["anderson", "mixed", "pse"])
    # solutes grow with the box; the crowded charged clusters need KH
    top = min(1500.0, max(30.0, n / 6000.0))
    atoms = int(round(math.exp(rng.uniform(math.log(6.0), math.log(top)))))
    if how in ("pse", "mixed"):
        atoms = min(atoms, 60 if how == "pse" else 300)
    c = _solve(None, grid, rng.choice([WATER, SALT, KCL]), atoms, rng.randint(24, 48),
               charge=float(rng.choice([0, 0, 1, -1])))
    if how == "anderson":
        c.update(anderson_m=rng.randint(3, 10), steps=rng.randint(16, 32))
    elif how == "mixed":
        # the first, plain FP32 phase, or the later blocks of difference-form
        # FP32 steps between FP64 steps
        c.update(precision=1, steps=rng.randint(5, 8), solvent=WATER, charge=0.0)
        if rng.random() < 0.5:
            c.update(mixed_switch=1e3, mixed_block=rng.randint(2, 4))
    elif how == "pse":
        c.update(closure="PSE3", solvent=WATER, charge=0.0, steps=rng.randint(12, 24))
    c["fields"] = n <= 300_000 and rng.random() < 0.4
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _closure(case):
    m = _package("rism3d")
    return {"KH": m.KH, "PSE3": m.PSE(3)}[case.get("closure", "KH")]


def _solute(case, seed):
    """A seeded solute, centred on its box as the .inp reader centres it."""
    G = _package("gen_inputs")
    n, q = case["atoms"], case.get("charge", 0.0)
    if n <= 60:
        s = G.random_walk_solute(n, seed, q)
    else:
        s = G.cluster_solute(n, (3.0 * n / (4.0 * math.pi * 0.1)) ** (1.0 / 3.0), seed, q)
    # PSE-3 runs away on such charges: it serves uncharged solutes (the -z switch)
    scale = 1.0 if case.get("closure", "KH") == "KH" else 0.0
    return _centred({"usig": s["sig"], "ueps": s["eps"], "uq": s["q"] * scale, "uxyz": s["xyz"]})


def _centred(s):
    mn, mx = s["uxyz"].min(0), s["uxyz"].max(0)
    return dict(s, uxyz=s["uxyz"] + np.floor(-(mx - mn) / 2 - mn + 0.5))


def _grid(case):
    return (case["nx"], case["ny"], case["nz"])


def _batch_inputs(case, seed):
    """[(grid, solute)] of a batch."""
    G = _package("gen_inputs")
    out = []
    for i in range(case["solutes"]):
        s = G.batch_solute(i, seed0=1_000_000 + 1000 * (int(seed) % 1_000_000))
        grid, _ = G.batch_grid(s["xyz"])
        out.append((grid, _centred({"usig": s["sig"], "ueps": s["eps"], "uq": s["q"],
                                    "uxyz": s["xyz"]})))
    return out


def _box(grid):
    return tuple(SPACING * g for g in grid)


def _solver(case, grid, solute):
    m = _package("rism3d")
    return m.RISM3D(grid, _box(grid), _solvent(case["solvent"]), solute, _closure(case),
                    anderson_m=case.get("anderson_m", 0), precision=case.get("precision", 0),
                    mixed_switch=case.get("mixed_switch", 0.0),
                    mixed_block=case.get("mixed_block", 0))


def _fields(case, seed):
    """Two short-ranged real fields like the c(r) that the solver transforms."""
    g = torch.Generator(device="cpu").manual_seed(int(seed))
    nx, ny, nz = _grid(case)
    out = []
    for _ in range(2):
        ax = []
        for n in (nz, ny, nx):
            r = (torch.arange(n, dtype=torch.float64) - n // 2) * SPACING
            x0 = (torch.rand(8, 1, generator=g, dtype=torch.float64) - 0.5) * 0.5 * n * SPACING
            ax.append(torch.exp(-(r[None, :] - x0) ** 2 / 4.0))
        a = torch.randn(8, generator=g, dtype=torch.float64)
        f = torch.einsum("i,iz,iy,ix->zyx", a, *ax)
        noise = torch.randn((ny, nx), generator=g, dtype=torch.float64)
        out.append(f + 1e-3 * noise)
    return out


def prepare(case, seed):
    k = case["kind"]
    if k == "solve":
        return {"case": case, "solver": _solver(case, _grid(case), _solute(case, seed))}
    if k == "batch":
        return {"case": case,
                "solvers": [_solver(case, g, s) for g, s in _batch_inputs(case, seed)]}
    if k == "analysis":
        g = _solver(case, _grid(case), _solute(case, seed))
        g.run(maxstep=case["steps"])
        return {"case": case, "solver": g}
    nx, ny, nz = _grid(case)
    f1, f2 = (f.cuda() for f in _fields(case, seed))
    half = (nz // 2, ny, nx)
    return {"case": case, "f1": f1, "f2": f2, "out": torch.empty_like(f1),
            "s1": torch.empty(half, dtype=torch.complex128, device="cuda"),
            "s2": torch.empty(half, dtype=torch.complex128, device="cuda")}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _thermo(th, single):
    """The .xmu quantities; of a solve that stops in its FP32 phase they are
    integrals of FP32 fields, and the values are returned in that type."""
    keep = ("SFE_SC", "SFEC_SC", "SFE_SC_HNC", "SFEC_SC_HNC", "SFE_GF", "SFEC_GF", "PMV",
            "Correction_Term")
    out = {k: th[k] for k in keep if th[k] is not None}
    return {k: np.asarray(v, np.float32) for k, v in out.items()} if single else out


def run(state):
    case = state["case"]
    m = _package("rism3d")
    if case["kind"] == "solve":
        g = state["solver"]
        th, _ = g.run(maxstep=case["steps"])
        out = _thermo(th, case["precision"] == 1)
        if case["fields"]:
            out["g"] = g.fields(m.FIELD_G)
            if case["precision"] == 1:
                out["g"] = out["g"].astype(np.float32)
        return out
    if case["kind"] == "batch":
        res = m.run_batch(state["solvers"], maxstep=case["steps"])
        ths = [_thermo(th, False) for th, _, _ in res]
        return {k: np.stack([np.asarray(t[k]) for t in ths]) for k in ths[0]}
    if case["kind"] == "analysis":
        g = state["solver"]
        return {"grad": g.analysis(m.ANALYSIS_GRAD), "euv": g.analysis(m.ANALYSIS_EUV)}
    grid, box = _grid(case), _box(_grid(case))
    stream = torch.cuda.current_stream().cuda_stream
    f1, f2, s1, s2, out = (state[k] for k in ("f1", "f2", "s1", "s2", "out"))
    m.fft_noalloc(-1, grid, box, f1.data_ptr(), s1.data_ptr(), stream)
    m.fft_noalloc(-1, grid, box, f2.data_ptr(), s2.data_ptr(), stream)
    m.fft_noalloc(+1, grid, box, out.data_ptr(), s2.data_ptr(), stream)
    return {"spectrum": s1, "back": out}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _solve_work(n_grid, sites, atoms, steps, anderson_m=0, words=8.0):
    """Words per step and grid point: t, u and fr read and the spectrum
    written (3n + 1), the spectrum read and written around the site-site
    product with fk (2n + 1), the spectrum, t, u and the history residuals
    read and R written (4n + hn), t, R and the mixed iterates read and t and
    one iterate written (4n + hn).  Set-up: u, fr, fk and t written, and the
    sums over the solute's atoms."""
    h = anderson_m or 2
    per = 13 * sites + 2 + 2 * h * sites
    nbytes = words * n_grid * per * steps + 8.0 * n_grid * (2 * sites + 2)
    fft = 2 * 2.5 * n_grid * math.log2(n_grid) * sites
    flops = steps * (fft + n_grid * (8 * sites * sites / 2 + 60 * sites))
    flops += float(n_grid) * atoms * (20 + 4 * sites) + 0.5 * n_grid * atoms * 8
    return nbytes, flops


def work(case):
    k = case["kind"]
    if k == "batch":
        b = f = 0.0
        for grid, s in _batch_inputs(case, 1):
            x, y = _solve_work(grid[0] * grid[1] * grid[2], 2, len(s["uq"]), case["steps"])
            b, f = b + x, f + y
        return {"bytes": b, "flops": f}
    n = case["nx"] * case["ny"] * case["nz"]
    if k == "transform":
        return {"bytes": 3 * 16.0 * n, "flops": 3 * 2.5 * n * math.log2(n)}
    sites = 2 if case["solvent"] == WATER else 4
    if k == "analysis":
        return {"bytes": 2 * 16.0 * n * sites, "flops": float(n) * sites * case["atoms"] * 50}
    b, f = _solve_work(n, sites, case["atoms"], case["steps"], case["anderson_m"],
                       4.0 if case["precision"] == 1 else 8.0)
    return {"bytes": b + (8.0 * n * sites if case["fields"] else 0.0), "flops": f}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
AVOGADRO, BOHR, BOLTZMANN, HARTREE = (6.02214076e23, 0.5291771500001, 1.380649e-23,
                                      4.359744722207185e-18)


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


class _Exact:
    """The solver's equations on the full complex grid with torch.fft."""

    def __init__(self, case, grid, solute):
        self.case, self.s, self.grid = case, _solvent(case["solvent"]), grid
        self.box = _box(grid)
        d = _dev()
        ten = lambda a: torch.as_tensor(np.asarray(a, np.float64), device=d)  # noqa: E731
        self.nv = int(self.s["natv"])
        self.q, self.rho = [float(x) for x in self.s["vq"]], [float(x) for x in self.s["vrho"]]
        nx, ny, nz = grid
        self.N, self.V = nx * ny * nz, self.box[0] * self.box[1] * self.box[2]
        self.dv = self.V / self.N
        self.r = [(torch.arange(n, dtype=torch.float64, device=d) - n // 2) * (b / n)
                  for n, b in zip(grid, self.box)]
        self.k = [2 * math.pi * (torch.arange(n, dtype=torch.float64, device=d) - n / 2.0 + 0.5) / b
                  for n, b in zip(grid, self.box)]
        # e^{-i k_j r_n} = out_j e^{-2 pi i j n / N} in_n
        self.pin, self.pout = [], []
        for n in grid:
            j = torch.arange(n, dtype=torch.float64, device=d)
            a = 0.5 - n / 2.0
            self.pin.append(torch.polar(torch.ones_like(j), -2 * math.pi * a * j / n))
            self.pout.append(torch.polar(torch.ones_like(j),
                                         math.pi * (j + a)))
        self.xyz, self.uq = ten(solute["uxyz"]), ten(solute["uq"])
        self.potentials(solute)
        self.chi()

    def phase(self, f, p):
        return f * p[2][:, None, None] * p[1][None, :, None] * p[0][None, None, :]

    def fwd(self, f):
        return self.dv * self.phase(torch.fft.fftn(self.phase(f.to(torch.complex128), self.pin)),
                                    self.pout)

    def inv(self, F):
        pc = [p.conj() for p in self.pout]
        ic = [p.conj() for p in self.pin]
        return (self.phase(torch.fft.ifftn(self.phase(F, pc)), ic) * (1.0 / self.dv)).real

    def potentials(self, solute):
        s, temper = self.s, float(self.s["temper"])
        ikbt = 1.0 / (AVOGADRO * BOLTZMANN * temper)
        ub = HARTREE * BOHR / (BOLTZMANN * temper)
        x, y, z = (self.r[0][None, None, :], self.r[1][None, :, None], self.r[2][:, None, None])
        shape = (self.grid[2], self.grid[1], self.grid[0])
        de, fr = (torch.zeros(shape, dtype=torch.float64, device=_dev()) for _ in range(2))
        lj = [torch.zeros_like(de) for _ in range(self.nv)]
        for a in range(len(self.uq)):
            px, py, pz = (float(v) for v in solute["uxyz"][a])
            q = float(solute["uq"][a])
            r2 = (x - px) ** 2 + (y - py) ** 2 + (z - pz) ** 2
            r = r2.sqrt()
            near = r < 1e-5
            ir = torch.where(near, torch.ones_like(r), r).reciprocal()
            de += torch.where(near, torch.zeros_like(r), q * ir)
            fr += torch.where(near, torch.full_like(r, q), -q * ir * torch.expm1(-r))
            for v in range(self.nv):
                sg = 0.5 * (float(solute["usig"][a]) + float(s["vsig"][v]))
                e4 = 4.0 * math.sqrt(float(solute["ueps"][a]) * float(s["veps"][v]))
                s6 = (r2 / (sg * sg)).clamp_(min=4e-6).pow_(-3)
                lj[v] += e4 * s6 * (s6 - 1.0)
        self.fr = fr * ub
        self.u = [lj[v] * ikbt + self.q[v] * (de * ub) for v in range(self.nv)]
        kx, ky, kz = self.k
        k2 = kx[None, None, :] ** 2 + ky[None, :, None] ** 2 + kz[:, None, None] ** 2
        e = [torch.polar(torch.ones((len(self.uq), len(k)), dtype=torch.float64, device=_dev()),
                         -self.xyz[:, d:d + 1] * k[None, :]) for d, k in enumerate(self.k)]
        ex = e[0] * self.uq[:, None]
        S = torch.empty(k2.shape, dtype=torch.complex128, device=_dev())
        for m in range(len(kz)):
            S[m] = (e[1] * e[2][:, m:m + 1]).t().contiguous() @ ex
        self.fk = S * (4 * math.pi * ub / (k2 * (k2 + 1.0)))
        self.k2 = k2

    def chi(self):
        """The natural cubic spline of the solvent's table at every |k|."""
        s, nt, nv = self.s, int(self.s["ntab"]), self.nv
        dk = math.pi / (float(s["dr"]) * nt)
        tab = dk * np.arange(1, nt + 1)
        kk = self.k2.sqrt()
        kmin, kmax = float(kk.min()), float(kk.max())
        below = np.nonzero(tab < kmin * (1 - 1e-12))[0]
        i0 = int(below[-1]) if len(below) else 0
        above = np.nonzero(tab > kmax * (1 + 1e-12))[0]
        i1 = int(above[0]) if len(above) else nt - 1
        xk = tab[i0:i1 + 1]
        yk = np.asarray(s["xvv"])[i0:i1 + 1].reshape(len(xk), -1)
        h = np.diff(xk)
        n = len(xk)
        sec = np.zeros_like(yk)  # second derivatives, zero at both ends
        diag, rhs = np.zeros(n), np.zeros_like(yk)
        for i in range(1, n - 1):
            d = 2.0 * (h[i - 1] + h[i])
            b = 6.0 * ((yk[i + 1] - yk[i]) / h[i] - (yk[i] - yk[i - 1]) / h[i - 1])
            if i > 1:
                w = h[i - 1] / diag[i - 1]
                d, b = d - w * h[i - 1], b - w * rhs[i - 1]
            diag[i], rhs[i] = d, b
        for i in range(n - 2, 0, -1):
            sec[i] = (rhs[i] - (h[i] * sec[i + 1] if i < n - 2 else 0.0)) / diag[i]
        c1, c2 = sec[:-1] / 2, (sec[1:] - sec[:-1]) / (6 * h[:, None])
        c0 = (yk[1:] - yk[:-1]) / h[:, None] - c1 * h[:, None] - c2 * h[:, None] ** 2
        ten = lambda a: torch.as_tensor(a, device=_dev())  # noqa: E731
        at = (torch.searchsorted(ten(xk), kk.reshape(-1), right=True) - 1).clamp_(0, n - 2)
        dx = kk.reshape(-1) - ten(xk)[at]
        self.X = []
        for pw in range(nv * nv):
            f = [ten(np.ascontiguousarray(a[:, pw]))[at] for a in (yk, c0, c1, c2)]
            self.X.append((((f[3] * dx + f[2]) * dx + f[1]) * dx + f[0]).reshape(kk.shape))

    def g_of(self, t, u):
        e = t - u
        kind = self.case.get("closure", "KH")
        up = 1 + e if kind == "KH" else 1 + e + e ** 2 / 2 + e ** 3 / 6
        return torch.where(e < 0, torch.exp(e.clamp(max=0.0)), up)

    def step(self):
        self.g = [self.g_of(t, u) for t, u in zip(self.t, self.u)]
        C = [self.fwd(g - 1 - t + q * self.fr) - q * self.fk
             for g, t, q in zip(self.g, self.t, self.q)]
        self.th = self.t
        self.R = []
        for v in range(self.nv):
            H = sum(self.X[v * self.nv + w] * C[w] for w in range(self.nv))
            self.R.append(self.inv(H) + 1 - self.g[v])

    def dot(self, a, b):
        return sum(float((x * y).sum()) / r for x, y, r in zip(a, b, self.rho))

    def solve(self, steps, count=2, beta=0.6, mp=0.2):
        """AN2 (two slots, the newest weighted by mp more) or Anderson(m)."""
        m = self.case.get("anderson_m", 0)
        self.t = [q * self.fr for q in self.q]
        sub = lambda a, b: [x - y for x, y in zip(a, b)]  # noqa: E731
        slot, hist, b = [None, None], [], 0
        for i in range(steps):
            self.step()
            R = self.R
            ss = sum(float((r * r).sum()) for r in R)
            if math.sqrt(ss / (self.N * self.nv)) <= 1e-6:  # converged: no further update
                break
            Q = [t + beta * r for t, r in zip(self.t, R)]
            old = hist if m else slot
            if i < count:
                new = [t + r for t, r in zip(self.t, R)]
            else:
                D = [sub(R, o[1]) for o in old]
                A = np.array([[self.dot(x, y) for y in D] for x in D])
                th = np.linalg.solve(A, np.array([self.dot(R, x) for x in D]))
                if not m:
                    th[1 - b] += mp
                new = [q + sum(c * (o[0][v] - q) for c, o in zip(th, old))
                       for v, q in enumerate(Q)]
            if m:
                hist = (hist + [(Q, R)])[-m:]
            else:
                slot[b], b = (Q, R), 1 - b
            self.t = new
        return self

    def thermo(self):
        s, kind = self.s, self.case.get("closure", "KH")
        ib = AVOGADRO * BOLTZMANN * float(s["temper"])
        sc, hnc, gf, cuv = [], [], [], 0.0
        for v in range(self.nv):
            t, th, u = self.t[v], self.th[v], self.u[v]
            h = self.R[v] + self.g[v] - 1
            eh, eg = h * 0.5 * t - (h - t), -(h * 0.5 + 1) * (h - t)
            e = eh
            if kind == "KH":
                e = torch.where(h > 0, eg, eh)
            elif kind == "PSE3":
                e = eh - (th - u).clamp(min=0.0) ** 4 / 24.0
            w = self.rho[v] * self.dv * ib
            sc.append(w * float(e.sum()))
            hnc.append(w * float(eh.sum()))
            gf.append(w * float(eg.sum()))
            cuv += self.rho[v] * self.dv * float((h - t).sum())
        xt = float(s["xt"])
        pmv = xt * (1 - cuv) * ib
        pres = 0.5 * (sum(self.rho) * 1e30 / AVOGADRO + 1 / (xt * ib))
        out = {"SFE_SC": sum(sc), "SFEC_SC": np.array(sc), "SFE_GF": sum(gf),
               "SFEC_GF": np.array(gf), "PMV": pmv * 1000.0, "Correction_Term": -pres * pmv * ib}
        if kind == "KH":
            out.update(SFE_SC_HNC=sum(hnc), SFEC_SC_HNC=np.array(hnc))
        return out

    def analysis(self, solute):
        """Per-atom forces (kcal/mol/A) and energies (J/mol)."""
        cc = HARTREE * BOHR * AVOGADRO
        x, y, z = (self.r[0][None, None, :], self.r[1][None, :, None], self.r[2][:, None, None])
        n = len(self.uq)
        grad, euv = np.zeros((n, 3)), np.zeros((n, 1 + self.nv))
        for a in range(n):
            px, py, pz = (float(v) for v in solute["uxyz"][a])
            dx, dy, dz = x - px, y - py, z - pz
            r2 = dx ** 2 + dy ** 2 + dz ** 2
            for v in range(self.nv):
                sg = 0.5 * (float(solute["usig"][a]) + float(self.s["vsig"][v]))
                eps = math.sqrt(float(solute["ueps"][a]) * float(self.s["veps"][v]))
                qq = cc * float(solute["uq"][a]) * self.q[v]
                w = torch.where(r2 >= (0.5 * sg) ** 2, self.g[v], torch.zeros_like(r2))
                i2 = torch.where(r2 > 0, r2, torch.ones_like(r2)).reciprocal()
                s6 = (sg * sg * i2) ** 3
                f = (24 * eps * s6 * i2 * (2 * s6 - 1) + qq * i2 * i2.sqrt()) * w
                for d, dd in enumerate((dx, dy, dz)):
                    grad[a, d] += self.rho[v] * float((f * dd).sum())
                e = (4 * eps * s6 * (s6 - 1) + qq * i2.sqrt()) * w
                euv[a, 1 + v] = self.dv * self.rho[v] * float(e.sum())
        euv[:, 0] = euv[:, 1:].sum(1)
        return {"grad": grad * self.dv / 4184.0, "euv": euv}


def exact(case, seed):
    k = case["kind"]
    if k == "transform":
        nx, ny, nz = _grid(case)
        f1, f2 = (f.to(_dev()) for f in _fields(case, seed))
        t = _Exact.__new__(_Exact)
        t.dv = SPACING ** 3
        t.pin, t.pout = [], []
        for n in (nx, ny, nz):
            j = torch.arange(n, dtype=torch.float64, device=_dev())
            a = 0.5 - n / 2.0
            t.pin.append(torch.polar(torch.ones_like(j), -2 * math.pi * a * j / n))
            t.pout.append(torch.polar(torch.ones_like(j), math.pi * (j + a)))
        return {"spectrum": t.fwd(f1)[nz // 2:].contiguous(), "back": f2}
    if k == "batch":
        res = [_Exact(case, g, s).solve(case["steps"]).thermo()
               for g, s in _batch_inputs(case, seed)]
        return {k: np.stack([np.asarray(r[k]) for r in res]) for k in res[0]}
    if case["nx"] * case["ny"] * case["nz"] > 20_000_000:
        return None  # minutes in plain torch
    solute = _solute(case, seed)
    e = _Exact(case, _grid(case), solute).solve(case["steps"])
    if k == "analysis":
        return e.analysis(solute)
    out = e.thermo()
    if case["fields"]:
        out["g"] = torch.stack(e.g).reshape(e.nv, -1)
    return out
