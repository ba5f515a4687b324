"""What the framework is timed on: MD steps, force evaluations, force-matching
gradients and batched replicas, through the public entry points.

Kinds of case (``case["kind"]``):

* ``md``     - ``Engine.step`` for ``steps`` steps, then the state a program
               writes to its trajectory (positions, velocities, accelerations)
               and the virial;
* ``forces`` - new positions in, ``Engine.recalculate``, accelerations and
               energies out (an outer integrator, a minimiser, Monte Carlo),
               with the potential and field at ``points`` places if asked;
* ``match``  - ``ForceMatcher.loss_and_grad`` over ``frames`` frames;
* ``batch``  - ``Batch.step`` for ``steps`` steps of ``replicas`` systems, then
               their positions and accelerations;
* ``grad``   - ``Batch.adjoint`` of ``replicas`` systems.

Fields (``case["fields"]``): ``lj`` (Lennard-Jones fluid), ``ions`` (+-1 ions,
LJ + Ewald), ``slab`` (ions between walls: Verlet-list LJ, short-range
Coulomb, Ewald_k in slab mode, ELC).  ``thermostat`` adds the temperature and
the Berendsen constraint of an equilibration run.
"""
import math

import numpy as np
import torch

from caviar_amd import Batch, Engine, configs, fitting
from caviar_amd.system import (BerendsenSettings, ELCSettings, EwaldKSettings, EwaldRSettings,
                               LJListSettings, LJSettings, NeighborSettings, ShortRangeSettings,
                               System, ThermoSettings)

COEF = 1.12347                       # cutoff_extra_coef of the ion workloads
THETA = (1.0, 0.8, 1.0, 1.2, 1.0, -1.0)   # force-matching target: eps, sigma, q of two species


# ------------------------------------------------------------------ cases --

def listed():
    return [
        # the smallest runs: a few hundred atoms, where launches and latency count
        dict(name="lj_256_fp64", kind="md", fields="lj", n=256, precision="fp64", steps=20),
        # a plain LJ fluid brought to temperature (the 4000-atom workload)
        dict(name="lj_4000_fp64_thermostat", kind="md", fields="lj", n=4000, precision="fp64",
             steps=50, thermostat=True),
        # the 8000-ion kmax 8 system in the plain form
        dict(name="ions_8000_fp64", kind="md", fields="ions", n=8000, precision="fp64", kmax=8,
             steps=20),
        # a production run of middle size, an atom count that fits no tile
        dict(name="ions_30011_mixed", kind="md", fields="ions", n=30011, precision="mixed", kmax=10,
             steps=20),
        # the headline workload: N = 262144, 32768 k-vectors
        dict(name="ions_262144_mixed", kind="md", fields="ions", n=262144, precision="mixed",
             kmax=16, steps=20),
        # the plain form where it is bound by the FP64 units
        dict(name="ions_65536_fp64", kind="md", fields="ions", n=65536, precision="fp64", kmax=12,
             steps=10),
        # forces, energies and a potential map of 100 ions at kmax 25
        dict(name="forces_100_fp64_points", kind="forces", fields="ions", n=100, precision="fp64",
             kmax=25, points=1000),
        # a force evaluation for an outer integrator
        dict(name="forces_100003_mixed", kind="forces", fields="ions", n=100003, precision="mixed",
             kmax=12, points=0),
        # ions between walls
        dict(name="forces_slab_3000_fp64", kind="forces", fields="slab", n=3000, precision="fp64",
             kmax=6, points=0),
        # one evaluation of the force-matching loss and its gradient
        dict(name="match_2000x8_fp64", kind="match", n=2000, precision="fp64", kmax=6, frames=8),
        # many small systems of one force field stepped together
        dict(name="batch_256_mixed", kind="batch", replicas=256, nmin=200, nmax=4000,
             precision="mixed", kmax=6, steps=50),
        # their force-matching gradients
        dict(name="grad_64_fp64", kind="grad", replicas=64, nmin=200, nmax=4000, precision="fp64",
             kmax=6),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["md", "md", "md", "forces", "forces", "match", "batch", "grad"])
    prec = rng.choice(["fp64", "mixed"])
    if kind == "md":
        if rng.random() < 0.35:
            return dict(kind="md", fields="lj", n=_log(rng, 256, 120000), precision=prec,
                        steps=rng.randint(5, 40), thermostat=rng.random() < 0.5)
        return dict(kind="md", fields="ions", n=_log(rng, 300, 262144 if prec == "mixed" else 65536),
                    precision=prec, kmax=rng.randint(4, 16 if prec == "mixed" else 12),
                    steps=rng.randint(4, 10))
    if kind == "forces":
        if rng.random() < 0.25:
            return dict(kind="forces", fields="slab", n=_log(rng, 300, 20000), precision=prec,
                        kmax=rng.randint(3, 8), points=0)
        n = _log(rng, 100, 150000)
        return dict(kind="forces", fields="ions", n=n, precision=prec,
                    kmax=rng.randint(4, 25 if n < 2000 else 12), points=rng.choice([0, _log(rng, 1, 5000)]))
    if kind == "match":
        return dict(kind="match", n=_log(rng, 300, 6000), precision=prec, kmax=rng.randint(4, 8),
                    frames=rng.randint(2, 12))
    if kind == "batch":
        return dict(kind="batch", replicas=_log(rng, 4, 256), nmin=200, nmax=4000, precision=prec,
                    kmax=rng.randint(4, 8), steps=rng.randint(4, 20))
    return dict(kind="grad", replicas=_log(rng, 4, 128), nmin=200, nmax=4000, precision=prec,
                kmax=rng.randint(4, 8))


# ----------------------------------------------------------------- inputs --

def _sites(n, box, dmin, rng):
    """n places in a periodic box (3 edges), no two closer than dmin: a random
    choice of the sites of a lattice, each displaced at random."""
    box = np.asarray(box, dtype=np.float64)
    m = np.maximum(1, np.round(box * (n / box.prod()) ** (1.0 / 3.0))).astype(int)
    while m.prod() < n:
        m[np.argmax(box / m)] += 1
    a = box / m
    at = rng.permutation(int(m.prod()))[:n]
    ix = np.stack([at % m[0], at // m[0] % m[1], at // (m[0] * m[1])], axis=1)
    amp = np.maximum(0.0, 0.5 * (a - dmin))
    return np.mod((ix + 0.5) * a + rng.uniform(-1, 1, (n, 3)) * amp, box)


def _ions(n, rho, kmax, rng, charge=(1.0, -1.0), parts=(0.5, 0.5)):
    box = (n / rho) ** (1.0 / 3.0)
    nt = len(charge)
    types = np.repeat(np.arange(nt), np.diff(np.round(np.cumsum((0.0,) + parts) * n).astype(int)))
    return System(lower=[0, 0, 0], upper=[box] * 3, bc=[1, 1, 1], ghost_cutoff=3.5 * COEF + 0.1,
                  mass=np.ones(nt), charge=charge, pos=_sites(n, [box] * 3, 0.8, rng),
                  vel=configs.maxwell_boltzmann(n, 1.0, np.ones(n), rng),
                  types=types[rng.permutation(n)],
                  neighbor=NeighborSettings(cutoff=3.5, cutoff_extra_coef=COEF),
                  lj=LJSettings(cutoff=2.5, epsilon=np.ones((nt, nt)), sigma=np.ones((nt, nt))),
                  ewald_r=EwaldRSettings(alpha=0.9, k_electrostatic=2.0),
                  ewald_k=EwaldKSettings.cube(0.9, kmax, 2.0))


def _lj(n, rng):
    box = (n / 0.8442) ** (1.0 / 3.0)
    return System(lower=[0, 0, 0], upper=[box] * 3, bc=[1, 1, 1], ghost_cutoff=2.9, mass=[1.0],
                  charge=[0.0], pos=_sites(n, [box] * 3, 0.9, rng),
                  vel=configs.maxwell_boltzmann(n, 0.72, np.ones(n), rng),
                  types=np.zeros(n, dtype=np.int32),
                  neighbor=NeighborSettings(cutoff=2.5, cutoff_extra_coef=2.8 / 2.5),
                  lj=LJSettings(cutoff=2.5, epsilon=np.ones((1, 1)), sigma=np.ones((1, 1))))


def _slab(n, kmax, rng):
    side = (n / 0.3 / 0.5) ** (1.0 / 3.0)
    height = 0.5 * side
    s = _ions(n, 0.3, kmax, rng)
    pos = _sites(n, [side, side, height - 1.0], 0.8, rng)
    pos[:, 2] += 0.5
    s = System(lower=[0, 0, 0], upper=[side, side, height], bc=[1, 1, 0], ghost_cutoff=s.ghost_cutoff,
               mass=s.mass, charge=s.charge, pos=pos, vel=s.vel, types=s.types, neighbor=s.neighbor,
               lj_list=LJListSettings(cutoff=2.5, epsilon_atom=np.ones(2), sigma_atom=np.ones(2)),
               short_range=ShortRangeSettings(cutoff=3.0, k_electrostatic=2.0),
               ewald_r=s.ewald_r,
               ewald_k=EwaldKSettings(alpha=0.9, k_electrostatic=2.0, kx_max=kmax, ky_max=kmax,
                                      kz_max=2 * kmax, slab_normal_axis=2, slab_lz=3.0 * height),
               elc=ELCSettings(slab_normal_axis=2, kx_max=4, ky_max=4, lz=3.0 * height,
                               k_electrostatic=2.0))
    return s


def _system(case, seed):
    rng = np.random.default_rng([int(seed), int(case["n"])])
    if case["fields"] == "lj":
        s = _lj(case["n"], rng)
    elif case["fields"] == "slab":
        s = _slab(case["n"], case["kmax"], rng)
    else:
        s = _ions(case["n"], 0.1 if case["n"] <= 100 else 0.3, case["kmax"], rng)
    if case.get("thermostat"):
        s.thermo = ThermoSettings(k_b=1.0)
        s.berendsen = BerendsenSettings(temperature=0.72, coupling=0.1, dt=_dt(case))
    return s, rng


def _replicas(case, seed):
    """Half-charged replicas; their sizes and densities belong to the case."""
    size = np.random.default_rng(case["replicas"])
    rng = np.random.default_rng([int(seed), int(case["replicas"])])
    return [_ions(int(size.integers(case["nmin"], case["nmax"] + 1)), size.uniform(0.2, 0.8),
                  case["kmax"], rng, charge=(1.0, -1.0, 0.0), parts=(0.25, 0.25, 0.5))
            for _ in range(case["replicas"])], rng


def _frames(case, seed):
    """Two species, `frames` configurations with the forces the target
    parameters give them, and a start up to a tenth off the target."""
    rng = np.random.default_rng([int(seed), int(case["n"]), int(case["frames"])])
    s = _ions(case["n"], 0.3, case["kmax"], rng)
    em, sm = fitting.mix(THETA[0:2], THETA[2:4])
    s.charge = np.array(THETA[4:6])
    s.lj.epsilon, s.lj.sigma = em, sm
    frames = np.stack([_sites(case["n"], s.size, 1.1, rng) for _ in range(case["frames"])])
    targets = np.stack([_Exact(s).forces(f).cpu().numpy() for f in frames])
    theta = np.asarray(THETA) * (1.0 + rng.uniform(-0.1, 0.1, 6))
    theta[5] = -theta[4]
    return fitting.FrameSet(s, frames, targets), theta


def _dt(case):
    return 0.005 if case.get("fields") == "lj" else 0.002


def prepare(case, seed):
    kind, prec = case["kind"], case["precision"]
    if kind == "match":
        fs, theta = _frames(case, seed)
        return dict(kind=kind, matcher=fitting.ForceMatcher(fs, precision=prec), theta=theta)
    if kind in ("batch", "grad"):
        systems, rng = _replicas(case, seed)
        b = Batch(systems, precision=prec)
        b.setup()
        w = [rng.normal(scale=1e-3, size=(s.n, 3)) for s in systems] if kind == "grad" else None
        return dict(kind=kind, batch=b, count=len(systems), steps=case.get("steps", 0), weights=w)
    s, rng = _system(case, seed)
    e = Engine(s, precision=prec)
    e.setup()
    if kind == "md":
        return dict(kind=kind, engine=e, dt=_dt(case), steps=case["steps"])
    new = s.pos + rng.uniform(-0.02, 0.02, s.pos.shape)
    return dict(kind=kind, engine=e, pos=new, slab=case["fields"] == "slab",
                points=rng.uniform(s.lower, s.upper, (case["points"], 3)) if case["points"] else None)


# -------------------------------------------------------------------- run --

def run(state):
    kind = state["kind"]
    if kind == "match":
        loss, grad = state["matcher"].loss_and_grad(state["theta"])
        return {"loss": loss, "grad": grad}
    if kind == "batch":
        b = state["batch"]
        b.step(0.002, state["steps"])
        return {w: np.concatenate([b.get(r, w) for r in range(state["count"])]) for w in ("pos", "acc")}
    if kind == "grad":
        g = state["batch"].adjoint(state["weights"])
        return {name: np.stack([x[k] for x in g]) for k, name in enumerate(("eps", "sigma", "charge"))}
    e = state["engine"]
    if kind == "md":
        e.step(state["dt"], state["steps"])
        return {"pos": e.get("pos"), "vel": e.get("vel"), "acc": e.get("acc"), "virial": e.virial()}
    e.set("pos", state["pos"])
    e.recalculate(force_rebuild=True)
    out = {"acc": e.get("acc"), "virial": e.virial()}
    if state["slab"]:
        out["elc"] = e.energy_elc()
        return out
    out["e_lj"], out["e_r"], out["e_k"] = e.energy()
    if state["points"] is not None:
        out["field_r"], out["pot_r"] = e.point_field("r", state["points"])
        out["field_k"], out["pot_k"] = e.point_field("k", state["points"])
    return out


# ------------------------------------------------------------- work, limits --

def _pass_flops(n, rho, kmax, fields):
    """One force evaluation: pairs within the list radius (43 operations for an
    Ewald pair, 12 for LJ) and the separable lattice sums."""
    if fields == "lj":
        return n * 0.5 * 4.18879 * 2.5 ** 3 * 0.8442 * 23
    pairs = n * 0.5 * 4.18879 * rho * (43 * (3.5 * COEF) ** 3 + 12 * 2.5 ** 3)
    kz = 2 * kmax if fields == "slab" else kmax
    rows, cols = (kmax + 1) * (2 * kmax + 1), 2 * kz + 1
    return pairs + n * rows * (6 + 8 * cols + 16 * cols + 22)


def work(case):
    kind = case["kind"]
    if kind in ("md", "forces"):
        n = case["n"]
        rho = 0.1 if n <= 100 else 0.3
        fl = _pass_flops(n, rho, case.get("kmax", 0), case["fields"])
        if kind == "md":  # positions, velocities, accelerations in and out of each step
            return {"bytes": 144.0 * n * case["steps"], "flops": (fl + 20.0 * n) * case["steps"]}
        rows, cols = (case["kmax"] + 1) * (2 * case["kmax"] + 1), 2 * case["kmax"] + 1
        return {"bytes": 48.0 * n + 56.0 * case["points"],
                "flops": fl + case["points"] * rows * (16 * cols + 22.0)}
    if kind == "match":  # forces and adjoint: about twice a force evaluation
        fl = _pass_flops(case["n"], 0.3, case["kmax"], "ions")
        return {"bytes": 96.0 * case["n"] * case["frames"], "flops": 2.0 * fl * case["frames"]}
    n = case["replicas"] * 0.5 * (case["nmin"] + case["nmax"])
    fl = _pass_flops(n, 0.5, case["kmax"], "ions")
    if kind == "batch":
        return {"bytes": 144.0 * n * case["steps"], "flops": (fl + 20.0 * n) * case["steps"]}
    return {"bytes": 48.0 * n, "flops": 1.5 * fl}


def tolerance(case):
    # fp64: 1e-15 of a force or gradient, 1e-13 of an acceleration after 50
    # steps of dynamics, more after several passes.  mixed: 5e-7 of a force
    # from its 32-bit pair and lattice terms (up to 7e-7 of the cancelling sums
    # of the virial), 6e-7 to 1e-6 after 10 to 20 steps; about four times that,
    # and room for the dynamics of several passes.
    moving = case["kind"] in ("md", "batch")
    if case["precision"] == "fp64":
        return {"rel": 1e-10 if moving else 1e-12}
    return {"rel": 2e-5 if moving else 4e-6}


# ------------------------------------------------------------------ exact --

class _Exact:
    """The same physics in 64 bits with plain torch: image atoms within
    ghost_cutoff past each face (one side per axis), pairs within the list
    radius at the last list build, shifted-force LJ, the real-space and
    lattice sums of Ewald."""

    def __init__(self, s):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.s = s
        self.lo, self.hi, self.L = (self.t(v) for v in (s.lower, s.upper, s.size))
        self.types = torch.as_tensor(s.types.astype(np.int64), device=self.dev)
        self.q = self.t(s.charge)
        self.eps, self.sig = (self.t(s.lj.epsilon), self.t(s.lj.sigma))
        self.rce = s.neighbor.cutoff * s.neighbor.cutoff_extra_coef
        self.old = None

    def t(self, a):
        return torch.as_tensor(np.asarray(a, dtype=np.float64), device=self.dev)

    def images(self, x):
        """Face flags and image atoms (source, shift in boxes) of wrapped positions."""
        gc = self.s.ghost_cutoff
        f = torch.where(x < self.lo + gc, -1, torch.where(x > self.hi - gc, 1, 0))
        src, shift = [], []
        for m in range(1, 8):
            on = torch.tensor([(m >> d) & 1 for d in range(3)], device=self.dev)
            i = torch.nonzero(((f != 0) | (on == 0)).all(1)).flatten()
            src.append(i)
            shift.append(-(f[i] * on).double())
        return f, torch.cat(src), torch.cat(shift)

    def pairs(self, x, src, shift):
        """Directed pairs (i, j, shift of j, j is an image) within the list radius."""
        n, r2 = len(x), self.rce ** 2
        y = torch.cat([x, x[src] + shift * self.L])
        owner = torch.cat([torch.arange(n, device=self.dev), src])
        sh = torch.cat([torch.zeros_like(x), shift])
        lo = y.min(0).values - 1e-9
        c = torch.floor((y - lo) / self.rce).long() + 1
        g = [int(v) + 2 for v in c.max(0).values]
        cell = (c[:, 0] * g[1] + c[:, 1]) * g[2] + c[:, 2]
        srt, perm = torch.sort(cell, stable=True)
        cnt = torch.bincount(srt, minlength=g[0] * g[1] * g[2])
        first = torch.cumsum(cnt, 0) - cnt
        out = []
        for k in range(27):
            off = ((k // 9 - 1) * g[1] + k // 3 % 3 - 1) * g[2] + k % 3 - 1
            nc, st = cnt[cell[:n] + off], first[cell[:n] + off]
            i = torch.repeat_interleave(torch.arange(n, device=self.dev), nc)
            j = torch.arange(len(i), device=self.dev) - (torch.cumsum(nc, 0) - nc)[i] + st[i]
            j = perm[j]
            d = y[j] - x[i]
            keep = ((d * d).sum(1) < r2) & (i != j)
            out.append((i[keep], j[keep]))
        i, j = (torch.cat([p[a] for p in out]) for a in (0, 1))
        return i, owner[j], sh[j], j >= n

    def build(self, x, force=False):
        """The list of wrapped positions x, rebuilt where the rebuild test asks for it."""
        f, src, shift = self.images(x)
        thr = 0.25 * (self.rce - self.s.neighbor.cutoff) ** 2
        if (force or self.old is None or not torch.equal(f, self.old[0])
                or bool((((x - self.old[1]) ** 2).sum(1) > thr).any())):
            self.list = self.pairs(x, src, shift)
            self.old = (f, x.clone())

    def short(self, x, energy=False):
        """Forces on each atom (and the virial, the LJ energy) from the list."""
        i, j, sh, ghost = self.list
        d = x[j] + sh * self.L - x[i]
        r2 = (d * d).sum(1)
        ti, tj = self.types[i], self.types[j]
        low = ghost | (i < j)   # the type matrices' row is the lower owned index
        a, b = torch.where(low, ti, tj), torch.where(low, tj, ti)
        rc2 = self.s.lj.cutoff ** 2
        near = (r2 <= rc2).double()
        e, g2 = self.eps[a, b], self.sig[a, b] ** 2
        s6, c6 = (g2 / r2) ** 3, (g2 / rc2) ** 3
        coef = 4 * e * near * ((6 * s6 - 12 * s6 * s6) / r2 + (12 * c6 * c6 - 6 * c6) / rc2)
        vir = torch.zeros((), dtype=torch.float64, device=self.dev)
        if self.s.ewald_r is not None:
            al, rn = self.s.ewald_r.alpha, torch.sqrt(r2)
            sr = (2 * al / math.sqrt(math.pi) * torch.exp(-al * al * r2)
                  + torch.special.erfc(al * rn) / rn) / r2
            ck = -self.s.ewald_r.k_electrostatic * self.q[ti] * self.q[tj] * sr
            vir = 0.5 * torch.sum(torch.where(i != j, -ck * r2, 0.0))
            coef = coef + ck
        f = torch.zeros_like(x).index_add(0, i, coef[:, None] * d)
        if not energy:
            return f, vir
        gc = (12 * c6 * c6 - 6 * c6) / rc2
        u = s6 * s6 - s6 + 0.5 * gc * r2 - (c6 * c6 - c6 + 0.5 * gc * rc2)
        return f, vir, 0.5 * torch.sum(4 * e * near * u)

    def lattice(self):
        """k along each axis and the weight f(k) of the vectors in use."""
        k = self.s.ewald_k
        ax = [torch.arange(-m, m + 1, device=self.dev, dtype=torch.float64) * (2 * math.pi) / float(l)
              for m, l in zip((k.kx_max, k.ky_max, k.kz_max), self.s.size)]
        k2 = (ax[0] ** 2)[:, None, None] + (ax[1] ** 2)[None, :, None] + (ax[2] ** 2)[None, None, :]
        f = torch.exp(-k2 / (4 * k.alpha ** 2)) / torch.where(k2 > 0, k2, 1.0)
        used = torch.cumsum((k2 > 0).flatten().long(), 0) <= 8 * k.kx_max * k.ky_max * k.kz_max
        return ax, torch.where((k2 > 0) & used.reshape(k2.shape), f, 0.0)

    def tables(self, x, ax):
        return [torch.exp(1j * x[:, d:d + 1] * ax[d][None, :]) for d in range(3)]

    def sk(self, x):
        ax, f = self.lattice()
        S = torch.zeros(f.shape[0] * f.shape[1], f.shape[2], dtype=torch.complex128, device=self.dev)
        for c in range(0, len(x), 16384):
            X, Y, Z = self.tables(x[c:c + 16384], ax)
            A = (self.q[self.types[c:c + 16384]][:, None, None] * X[:, :, None] * Y[:, None, :])
            S = S + A.reshape(len(X), -1).T.contiguous() @ Z
        return ax, f, S.reshape(f.shape)

    def long(self, p, ax, f, S):
        """Field and potential of the lattice sum at places p."""
        k = self.s.ewald_k
        c0 = 4 * math.pi * k.k_electrostatic / float(np.prod(self.s.size))
        T = torch.conj(f * S)
        G = torch.stack([T, T * ax[0][:, None, None], T * ax[1][None, :, None], T * ax[2][None, None, :]])
        G = G.permute(3, 0, 1, 2).reshape(len(ax[2]), -1).contiguous()
        out = []
        for c in range(0, len(p), 4096):
            X, Y, Z = self.tables(p[c:c + 4096], ax)
            U = (Z @ G).reshape(len(X), 4, -1)
            P = (X[:, :, None] * Y[:, None, :]).reshape(len(X), 1, -1)
            out.append((U * P).sum(2))
        v = c0 * torch.cat(out)
        return v[:, 1:].imag, v[:, 0].real

    def forces(self, pos):
        """Forces of the wrapped positions (list rebuilt), differentiable in eps, sig, q."""
        x = torch.remainder(self.t(pos) - self.lo, self.L) + self.lo
        self.build(x, force=True)
        f = self.short(x)[0]
        if self.s.ewald_k is not None:
            f = f + self.q[self.types][:, None] * self.long(x, *self.sk(x))[0]
        return f

    def acc(self, x):
        f, vir = self.short(x)
        if self.s.ewald_k is not None:
            f = f + self.q[self.types][:, None] * self.long(x, *self.sk(x))[0]
        return f, vir     # unit masses

    def wrap(self, x):
        up, dn = x < self.lo, x > self.hi
        return x + self.L * up - self.L * dn, bool((up | dn).any())

    def run(self, dt, steps):
        s = self.s
        x, v = self.wrap(self.t(s.pos))[0], self.t(s.vel)
        self.build(x, force=True)
        a, vir = self.acc(x)
        for _ in range(steps):
            x, wrapped = self.wrap(x + v * dt + 0.5 * a * dt * dt)
            self.build(x, force=wrapped)
            b, vir = self.acc(x)
            v, a = v + 0.5 * dt * (a + b), b
            if s.berendsen is not None:
                t = ((v - v.mean(0)) ** 2).sum() / (s.thermo.k_b * (3 * s.n - 3))
                bs = s.berendsen
                lam = torch.sqrt(1.0 + bs.dt / bs.coupling * (bs.temperature / t - 1.0))
                v = v * torch.clamp(lam, bs.lambda_min, bs.lambda_max)
        return x, v, a, vir

    def grad(self, pos, w):
        """d/d(eps, sigma, q) of sum_i w_i . F_i."""
        par = [v.clone().requires_grad_(True) for v in (self.eps, self.sig, self.q)]
        self.eps, self.sig, self.q = par
        f = self.forces(pos)
        g = torch.autograd.grad((f * self.t(w)).sum(), par)
        return f.detach(), g


def _np(*tensors):
    return [t.detach().cpu().numpy() for t in tensors]


def exact(case, seed):
    kind = case["kind"]
    if kind == "match":
        fs, theta = _frames(case, seed)
        loss, ge, gs, gq = 0.0, 0.0, 0.0, 0.0
        em, sm = _mix(theta)
        scale = 1.0 / (len(fs.frames) * case["n"] * 3)
        for pos, target in zip(fs.frames, fs.targets):
            e = _Exact(fs.system)
            e.eps, e.sig, e.q = e.t(em), e.t(sm), e.t(theta[4:6])
            r = (e.forces(pos) - e.t(target)).detach()
            loss += scale * float((r * r).sum())
            _, g = e.grad(pos, (2 * scale * r).cpu().numpy())
            ge, gs, gq = (a + b.cpu().numpy() for a, b in zip((ge, gs, gq), g))
        de, ds = _mix_gradient(theta, em, ge, gs)
        return {"loss": loss, "grad": np.concatenate([de, ds, gq])}
    if kind in ("batch", "grad"):
        systems, rng = _replicas(case, seed)
        if kind == "batch":
            if sum(s.n for s in systems) * case["steps"] > 1_500_000:
                return None
            got = [_np(*_Exact(s).run(0.002, case["steps"])) for s in systems]
            return {"pos": np.concatenate([g[0] for g in got]), "acc": np.concatenate([g[2] for g in got])}
        w = [rng.normal(scale=1e-3, size=(s.n, 3)) for s in systems]
        got = [_np(*_Exact(s).grad(s.pos, u)[1]) for s, u in zip(systems, w)]
        return {name: np.stack([g[k] for g in got]) for k, name in enumerate(("eps", "sigma", "charge"))}
    if case["fields"] == "slab":
        return None
    s, rng = _system(case, seed)
    e = _Exact(s)
    if kind == "md":
        if s.n * case["steps"] > 3_000_000:
            return None
        x, v, a, vir = _np(*e.run(_dt(case), case["steps"]))
        return {"pos": x, "vel": v, "acc": a, "virial": float(vir)}
    new = s.pos + rng.uniform(-0.02, 0.02, s.pos.shape)
    pts = rng.uniform(s.lower, s.upper, (case["points"], 3)) if case["points"] else None
    x = e.wrap(e.t(new))[0]
    e.build(x, force=True)
    f, vir, elj = e.short(x, energy=True)
    lat = e.sk(x)
    f = f + e.q[e.types][:, None] * e.long(x, *lat)[0]
    k = s.ewald_k
    ek = (0.5 * 4 * math.pi * k.k_electrostatic / float(np.prod(s.size))
          * float((lat[1] * lat[2].abs() ** 2).sum())
          - k.alpha / math.sqrt(math.pi) * k.k_electrostatic * float((e.q[e.types] ** 2).sum()))
    # the real-space energy and point sums take every atom of 27 cells, which
    # only the cell walk itself defines
    out = {"acc": _np(f)[0], "virial": float(vir), "e_lj": float(elj), "e_r": None, "e_k": ek}
    if pts is not None:
        out["field_r"] = out["pot_r"] = None
        out["field_k"], out["pot_k"] = _np(*e.long(e.t(pts), *lat))
    return out


def _mix(theta):
    """Lorentz-Berthelot matrices of two species."""
    e, s = np.asarray(theta[0:2]), np.asarray(theta[2:4])
    return np.sqrt(np.outer(e, e)), 0.5 * (s[:, None] + s[None, :])


def _mix_gradient(theta, em, ge, gs):
    """Matrix gradients chained to the species' values."""
    e = np.asarray(theta[0:2])
    de = ((ge + ge.T) * em).sum(1) / (2.0 * e)
    return de, 0.5 * (gs + gs.T).sum(1)
