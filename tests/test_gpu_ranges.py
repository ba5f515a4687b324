"""Kernels at the sizes where their work splits change: edges of tiles and
chunks, remainders, the smallest and largest of a range.

FP64 results are compared with the oracle at 1e-12 relative (norm-wise): sums
of at most a few thousand terms in another order differ by about
sqrt(terms) * 1e-16 of the terms' size, and the terms here do not cancel by
more than 1e3.
"""
import numpy as np
import pytest

import fixtures as F
from caviar_amd import Batch, Engine, NaNAccelerationError, configs
from oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,rho,coef", [(1, 0.01, 1.12347), (5, 0.02, 1.12347), (61, 0.1, 1.3),
                                        (700, 0.3, 1.12347), (1500, 0.8, 1.12347)])
@pytest.mark.parametrize("pair_kernel", ["auto", "rows"])
def test_cell_walk_energies_and_points(gpu, n, rho, coef, pair_kernel):
    """Real-space energy, LJ energy and real-space point sums: from one atom to
    stencils of several staging passes (over 512 candidates), point counts off
    the wave size, a point on an atom."""
    print(f"[case] cell walk n={n} rho={rho} {pair_kernel}", flush=True)
    s = configs.ions(n=n, rho=rho, kmax=2, seed=n, coef=coef)
    o = Oracle(s)
    o.setup()
    e = Engine(s)
    e.set_pair_kernel(pair_kernel)
    e.setup()
    elj, er, _ = e.energy()
    assert abs(er - o.energy_r()) <= 1e-12 * abs(o.energy_r())
    assert abs(elj - o.energy_lj()) <= 1e-12 * max(abs(o.energy_lj()), 1e-300)
    rng = np.random.default_rng(3)
    for np_ in (1, 65, 258):
        pts = rng.uniform(s.lower, s.upper, (np_, 3))
        pts[0] = s.pos[0]
        f, p = e.point_field("r", pts)
        fo, po = o.point_r(pts)
        assert F.rel_err(f, fo) <= 1e-12
        assert F.rel_err(p, po) <= 1e-12


@pytest.mark.parametrize("n,k", [(1, (1, 1, 1)), (127, (2, 3, 4)), (129, (9, 9, 9)), (300, (25, 25, 25)),
                                 (900, (3, 3, 40)), (4100, (6, 6, 6))])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_force_pass_row_splits(gpu, n, k, precision):
    """Lattice forces and point fields where the row blocks of the force pass
    are split over workgroups (few atoms, long lattices, two K slabs), against
    the oracle.  Mixed: 32-bit sums, 1e-5 of the force RMS."""
    print(f"[case] force splits n={n} k={k} {precision}", flush=True)
    s = configs.ions(n=n, rho=0.3 if n > 1 else 0.01, kmax=1, seed=n, with_lj=False, with_r=False)
    s.neighbor = None
    s.ewald_k.kx_max, s.ewald_k.ky_max, s.ewald_k.kz_max = k
    o = Oracle(s)
    o.setup()
    e = Engine(s, precision=precision)
    e.setup()
    tol = 1e-12 if precision == "fp64" else 1e-5
    a = o.get("acc")
    if n > 1:
        assert F.rel_err(e.get("acc"), a) <= tol
    pts = np.random.default_rng(1).uniform(s.lower, s.upper, (131, 3))
    f, p = e.point_field("k", pts)
    fo, po = o.point_k(pts)
    assert F.rel_err(f, fo) <= tol
    assert F.rel_err(p, po) <= tol


def _free_pair_system(n, box, pos, vel, rce=2.0):
    """Neutral atoms with an LJ reach of 0.2: they fly straight until two meet."""
    from caviar_amd import LJSettings, NeighborSettings, System
    return System(lower=[0, 0, 0], upper=[box] * 3, bc=[1, 1, 1], ghost_cutoff=rce + 0.1, mass=[1.0],
                  charge=[0.0], pos=pos, vel=vel, types=np.zeros(n, dtype=np.int32),
                  neighbor=NeighborSettings(cutoff=rce / 1.25, cutoff_extra_coef=1.25),
                  lj=LJSettings(cutoff=0.2, epsilon=np.ones((1, 1)), sigma=np.full((1, 1), 0.1)))


@pytest.mark.parametrize("steps", [5, 20, 70])
def test_nan_among_queued_steps(gpu, steps):
    """Two atoms meet exactly in step 4: the NaN shows at the start of step 5,
    and the state is that before it however many steps were asked for."""
    print(f"[case] queued NaN steps={steps}", flush=True)
    pos = np.array([[4.0, 5.0, 5.0], [6.0, 5.0, 5.0], [1.0, 1.0, 1.0]])
    vel = np.array([[2.0, 0.0, 0.0], [-2.0, 0.0, 0.0], [0.25, 0.5, 0.0]])
    s = _free_pair_system(3, 16.0, pos, vel)
    e = Engine(s)
    e.setup()
    with pytest.raises(NaNAccelerationError):
        e.step(0.125, steps)
    want = pos + 4 * 0.125 * vel
    assert np.array_equal(e.get("pos"), want)
    assert np.isnan(e.get("acc")[:2]).all() and not np.isnan(e.get("acc")[2]).any()
    # the atoms moved apart again: the run goes on
    want[1, 1] += 1.0
    e.set("pos", want)
    e.set("vel", vel)
    e.recalculate()
    e.step(0.125, 3)
    assert np.array_equal(e.get("pos"), want + 3 * 0.125 * vel)


@pytest.mark.parametrize("steps", [1, 7, 80])
def test_list_overflow_among_queued_steps(gpu, steps):
    """Atoms flying together outgrow the list rows (sized for the mean density)
    and the cell buckets in the middle of a run; the trajectory is the
    oracle's, the pairs the exact set."""
    print(f"[case] queued overflow, {steps} steps a call", flush=True)
    rng = np.random.default_rng(11)
    n, box = 400, 40.0
    end = np.array([20.5, 20.5, 20.5]) + rng.uniform(-0.9, 0.9, (n, 3))
    pos = rng.uniform(0.5, box - 0.5, (n, 3))
    dt, total = 1.0 / 128, 80
    vel = (end - pos) / (dt * 76)
    s = _free_pair_system(n, box, pos, vel)
    s.lj.epsilon[:] = 0.0
    o = Oracle(s)
    o.setup()
    assert o.run(dt, total) == 0
    e = Engine(s)
    e.setup()
    left = total
    while left:
        k = min(steps, left)
        e.step(dt, k)
        left -= k
    assert F.rel_err(e.get("pos"), o.get("pos")) <= 1e-12
    assert np.array_equal(F.sorted_pairs(e.pairs()), F.sorted_pairs(o.pairs()))


@pytest.mark.parametrize("clump", [1, 60, 66, 130, 700])
def test_crowded_cells(gpu, clump):
    """Cells from empty to far past their buckets (sorted through memory):
    ghosts and pairs bit-exact, forces against the oracle."""
    print(f"[case] crowded cell {clump}", flush=True)
    rng = np.random.default_rng(clump)
    n, box = clump + 150, 30.0
    pos = rng.uniform(0, box, (n, 3))
    pos[rng.permutation(n)[:clump]] = rng.uniform(13.0, 14.9, (clump, 3))
    s = configs.ions(n=n, rho=n / box ** 3, kmax=1, seed=1, dmin=0.0, with_lj=False, with_k=False)
    s.pos = np.ascontiguousarray(pos)
    o = Oracle(s)
    o.setup()
    e = Engine(s)
    e.setup()
    gp, gs = e.ghosts()
    og, os_ = o.ghost_data()
    assert np.array_equal(gp, og) and np.array_equal(gs, os_)
    assert np.array_equal(F.sorted_pairs(e.pairs()), F.sorted_pairs(o.pairs()))
    assert F.rel_err(e.get("acc"), o.get("acc")) <= 1e-11  # close pairs cancel more


@pytest.mark.parametrize("clump", [60, 66, 130, 700, 1500])
def test_crowded_cells_again(gpu, clump):
    """Once crowded cells were met their buckets grow: the builds after that
    sort them from the bucket, in an engine and in a batch (beside a replica
    that is not crowded).  Free atoms that drift together: positions exactly,
    pairs the exact set after every few steps."""
    print(f"[case] crowded cells again {clump}", flush=True)
    rng = np.random.default_rng(clump)
    n, box, dt = clump + 150, 24.0, 0.0625
    pos = rng.uniform(0, box, (n, 3))
    pos[rng.permutation(n)[:clump]] = rng.uniform(12.0, 13.9, (clump, 3))
    pos = np.round(pos * 1024) / 1024       # the drift is exact
    s = _free_pair_system(n, box, pos, np.tile([3.0, -1.0, 0.5], (n, 1)))
    s.lj.epsilon[:] = 0.0
    other = _free_pair_system(50, box, np.round(rng.uniform(0, box, (50, 3)) * 1024) / 1024,
                              np.zeros((50, 3)))
    e, b = Engine(s.copy()), Batch([s, other])
    e.setup()
    b.setup()
    now = pos
    for steps in (1, 1, 5, 9):
        e.step(dt, steps)
        b.step(dt, steps)
        for _ in range(steps):
            now = now + s.vel * dt
            now = np.where(now < 0, now + box, np.where(now > box, now - box, now))
        assert np.array_equal(e.get("pos"), now) and np.array_equal(b.get(0, "pos"), now)
        assert np.array_equal(F.sorted_pairs(e.pairs()), F.sorted_pairs(b.pairs(0)))
    e.recalculate(force_rebuild=True)
    gp, _ = F.numpy_ghosts(s, now)
    assert np.array_equal(F.sorted_pairs(e.pairs()), F.sorted_pairs(F.exact_pairs(now, gp, 2.0)))


@pytest.mark.parametrize("n", [63, 64, 65, 257, 16383, 16385])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_steps_at_workgroup_edges(gpu, n, precision):
    """Atom counts about the sizes where workgroups, lanes per atom and waves
    per cell change: 12 steps, list kept and rebuilt, against the oracle
    (1e-9 after the steps; mixed 1e-5), ghosts and pairs exactly."""
    print(f"[case] steps n={n} {precision}", flush=True)
    s = configs.ions(n=n, rho=0.3, kmax=2, seed=n)
    o = Oracle(s, threads=8)
    o.setup()
    assert o.run(0.002, 12) == 0
    e = Engine(s, precision=precision)
    e.setup()
    e.step(0.002, 5)
    e.step(0.002, 7)
    tol = 1e-9 if precision == "fp64" else 1e-5
    for what in ("pos", "vel", "acc"):
        assert F.rel_err(e.get(what), o.get(what)) <= tol, what
    if precision == "fp64":
        assert abs(e.virial() - o.virial()) <= 1e-9 * abs(o.virial())
        assert np.array_equal(F.sorted_pairs(e.pairs()), F.sorted_pairs(o.pairs()))


@pytest.mark.parametrize("n,kmax,types", [(2, 1, 2), (33, 3, 1), (700, 7, 3), (3000, 16, 4), (9000, 4, 2)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_adjoint_weight_sets(gpu, n, kmax, types, precision):
    """The adjoint's structure factors, all weight sets of a launch at once (and
    in several launches where their partials are large), against the oracle's:
    1e-10 (FP64; the gradient cancels sums 100 times its size), mixed 1e-4."""
    print(f"[case] weight sets n={n} kmax={kmax} types={types} {precision}", flush=True)
    s = configs.ions(n=n, rho=0.3 if n > 2 else 0.02, kmax=kmax, seed=n)
    rng = np.random.default_rng(n)
    s.mass = np.ones(types)
    s.charge = rng.uniform(-1, 1, types)
    s.types = rng.integers(0, types, n).astype(np.int32)
    s.lj.epsilon = np.ones((types, types))
    s.lj.sigma = rng.uniform(0.8, 1.1, (types, types))
    o = Oracle(s, threads=8)
    o.setup()
    e = Engine(s, precision=precision)
    e.setup()
    w = rng.normal(size=(n, 3))
    tol = 1e-10 if precision == "fp64" else 1e-4
    for a, b in zip(e.adjoint(w), o.adjoint(w)):
        assert F.rel_err(np.ravel(a), np.ravel(b)) <= tol


@pytest.mark.parametrize("alpha", [0.9, 2.5, 0.0])
def test_real_space_terms_accuracy(gpu, alpha):
    """Potential and field of one ion at distances from 1e-3 to 1.4 cells
    (alpha r from 0 to 10), against 40-digit erfc and exp: 4e-15 relative, i.e.
    8 ulp for the fit at large alpha r and 10 for the distance, the products and
    the exponential's last bit."""
    mp = pytest.importorskip("mpmath")
    mp.mp.dps = 40
    print(f"[case] real-space terms alpha={alpha}", flush=True)
    s = configs.ions(n=1, rho=1e-3, kmax=1, seed=1, with_lj=False, with_k=False)
    s.lower, s.upper = np.zeros(3), np.full(3, 64.0)
    s.bc = np.zeros(3, dtype=np.int32)
    s.pos = np.array([[32.0, 32.0, 32.0]])
    s.ewald_r.alpha, s.ewald_r.k_electrostatic = alpha, 1.0
    e = Engine(s)
    e.setup()
    # distances exact in FP64 differences: multiples of 2^-20
    r = np.unique(np.round(np.geomspace(1e-3, 4.0, 400) * 2 ** 20) / 2 ** 20)
    pts = np.repeat(s.pos, len(r), axis=0)
    pts[:, 0] += r
    f, p = e.point_field("r", pts)
    q = float(s.charge[s.types[0]])
    al = mp.mpf(alpha)
    for k in range(len(r)):
        x = mp.mpf(float(r[k]))
        ec = mp.erfc(al * x) / x
        g = (2 * al / mp.sqrt(mp.pi) * mp.exp(-(al * x) ** 2) + ec) / x
        if ec < mp.mpf(10) ** -290:
            continue
        assert abs(mp.mpf(float(p[k])) - q * ec) <= 4e-15 * abs(ec), (r[k], alpha)
        assert abs(mp.mpf(float(f[k, 0])) - q * g) <= 4e-15 * abs(g), (r[k], alpha)


def test_real_space_terms_rounding(gpu):
    """The same terms' usual error, where alpha r is small and they are largest:
    about ten roundings between the distance and each sum, of at most
    2^-53 / sqrt(3) = 6.4e-17 root mean square each, so 2e-16; the distance's
    square counts up to 1.4 times (alpha^2 r^2)."""
    mp = pytest.importorskip("mpmath")
    mp.mp.dps = 40
    print("[case] real-space terms' rounding", flush=True)
    s = configs.ions(n=1, rho=1e-3, kmax=1, seed=1, with_lj=False, with_k=False)
    s.lower, s.upper = np.zeros(3), np.full(3, 64.0)
    s.bc = np.zeros(3, dtype=np.int32)
    s.pos = np.array([[32.0, 32.0, 32.0]])
    s.ewald_r.alpha, s.ewald_r.k_electrostatic = 0.3, 1.0
    e = Engine(s)
    e.setup()
    pts = np.repeat(s.pos, 1500, axis=0)
    pts[:, 0] += np.random.default_rng(5).uniform(0.7, 4.0, len(pts))
    f, p = e.point_field("r", pts)
    q = float(s.charge[s.types[0]])
    al = mp.mpf(0.3)
    err = np.empty((2, len(pts)))
    for k in range(len(pts)):
        x = mp.mpf(float(pts[k, 0])) - 32
        ec = mp.erfc(al * x) / x
        g = (2 * al / mp.sqrt(mp.pi) * mp.exp(-(al * x) ** 2) + ec) / x
        err[0, k] = float(mp.mpf(float(p[k])) / (q * ec) - 1)
        err[1, k] = float(mp.mpf(float(f[k, 0])) / (q * g) - 1)
    rms = np.sqrt((err ** 2).mean(1))
    assert rms[0] <= 2e-16 and rms[1] <= 2e-16, rms


@pytest.mark.parametrize("n", [255, 256, 700])
@pytest.mark.parametrize("n_r_df,which", [(d, w) for d in (0, 3) for w in
                                          ("temp", "berendsen", "nve", "both", "both_no_temp")]
                         + [(5, "temp")])   # the kinetic energy is 0 there: no finite factors
def test_constraints_end_of_step(gpu, n, n_r_df, which):
    """A step's end with every combination of temperature, Berendsen, NVE and
    pressure, against the oracle after 6 steps (1e-9), with atom counts about a
    block of partial sums."""
    from caviar_amd import BerendsenSettings, NVESettings, ThermoSettings
    print(f"[case] constraints n={n} n_r_df={n_r_df} {which}", flush=True)
    s = configs.ions(n=n, rho=0.3, kmax=2, seed=n)
    s.thermo = ThermoSettings(k_b=1.3, n_r_df=n_r_df, temperature_process=which != "both_no_temp",
                              pressure_process=True)
    if which in ("berendsen", "both", "both_no_temp"):
        s.berendsen = BerendsenSettings(temperature=0.9, coupling=0.05, dt=0.002, step=2)
    if which in ("nve", "both", "both_no_temp"):
        s.nve = NVESettings(kbt=1.1, step=3)
    o = Oracle(s)
    o.setup()
    assert o.run(0.002, 6) == 0
    e = Engine(s)
    e.setup()
    e.step(0.002, 6)
    assert F.rel_err(e.get("vel"), o.get("vel")) <= 1e-9
    for got, want in zip(e.thermo(), o.thermo()):
        assert abs(got - want) <= 1e-9 * abs(want)


def _exchange_replicas():
    rng = np.random.default_rng(8)

    def free(n, box, pos):
        return _free_pair_system(n, box, np.ascontiguousarray(pos), rng.normal(scale=3.0, size=(n, 3)))

    face = rng.uniform(0, 6.0, (41, 3))       # the box is three cells: the upper faces
    face[:7, 0] = 6.0                         # lie in the layer past the inner cells
    face[5:12, 1] = 6.0
    face[6] = 6.0
    crowd = rng.uniform(0, 12.0, (700, 3))
    # 600 atoms in one cell, 0.21 apart: beyond the LJ reach at the start and
    # hardly into it after 12 steps (0.07 each), so that no collision amplifies
    # the order of the sums
    g = np.stack(np.meshgrid(*[np.arange(9) * 0.211 + 4.1] * 3, indexing="ij"), -1).reshape(-1, 3)
    crowd[:600] = g[rng.permutation(len(g))[:600]]
    out = [free(41, 6.0, face), free(700, 12.0, crowd), free(40, 90.0, rng.uniform(0, 90.0, (40, 3))),
           free(1, 4.5, [[4.4, 0.1, 2.0]])]
    out += [free(n, 9.0, rng.uniform(0, 9.0, (n, 3))) for n in (255, 256, 257)]
    # atoms that leave the middle of their box: images beyond the slots set aside
    g = np.stack(np.meshgrid(*[np.arange(7) * 0.5 + 6.5] * 3, indexing="ij"), -1).reshape(-1, 3)
    s = free(len(g), 16.0, g)
    s.vel = np.ascontiguousarray((g - 8.0) * 150.0)
    return out + [s]


@pytest.mark.parametrize("which", ["all", "fixed", "face"])
def test_batch_exchange_edges(gpu, which):
    """Images, cells and rows of a batch: atoms on the upper faces, cells past
    their buckets, more cells than a workgroup adds up itself, one atom, counts
    about the workgroup, ghosts outgrowing their slots.  Pairs exactly as the
    oracle's, positions within 1e-12 after 12 steps."""
    print(f"[case] batch exchange {which}", flush=True)
    systems = _exchange_replicas()
    systems = {"all": systems, "fixed": systems[:-1], "face": systems[:1]}[which]
    b = Batch(systems)
    b.setup()
    for r, s in enumerate(systems):
        o = Oracle(s.copy())
        o.setup()
        assert np.array_equal(F.sorted_pairs(b.pairs(r)), F.sorted_pairs(o.pairs())), r
        e = Engine(s.copy())
        e.setup()
        assert np.array_equal(F.sorted_pairs(e.pairs()), F.sorted_pairs(o.pairs())), r
    b.step(0.002, 12)
    for r, s in enumerate(systems):
        o = Oracle(s.copy())
        o.setup()
        assert o.run(0.002, 12) == 0
        assert F.rel_err(b.get(r, "pos"), o.get("pos")) <= 1e-12, r
        if which != "all":  # (a replica outgrowing its slots has every list rebuilt)
            assert np.array_equal(F.sorted_pairs(b.pairs(r)), F.sorted_pairs(o.pairs())), r


@pytest.mark.parametrize("n", [333, 17000])
@pytest.mark.parametrize("ids", ["ascending", "gaps", "shuffled", "equal"])
@pytest.mark.parametrize("symmetric", [True, False])
def test_pair_rows_by_ids(gpu, n, ids, symmetric):
    """The row kernel tells images and the order of a pair by ids that ascend
    with the index, else by the slots' atoms: forces and virial for both, with
    type tables that depend on which atom is the lower one."""
    print(f"[case] ids {ids} n={n} symmetric={symmetric}", flush=True)
    s = configs.ions(n=n, rho=0.3, kmax=1, seed=n, with_k=False)
    rng = np.random.default_rng(n)
    s.ids = {"ascending": np.arange(n), "gaps": np.cumsum(rng.integers(1, 5, n)),
             "shuffled": rng.permutation(n), "equal": np.full(n, 7)}[ids].astype(np.int32)
    if not symmetric:
        s.lj.epsilon = np.array([[1.0, 0.7], [1.3, 0.9]])
        s.lj.sigma = np.array([[1.0, 0.95], [1.05, 0.9]])
    o = Oracle(s, threads=8)
    o.setup()
    for kernel in ("auto", "rows"):
        e = Engine(s)
        e.set_pair_kernel(kernel)
        e.setup()
        assert F.rel_err(e.get("acc"), o.get("acc")) <= 1e-12, kernel
        # the oracle adds some 38 n terms one by one: a random walk of the roundings
        # of partial sums that reach 41 times the total (n = 17000, counted),
        # 1.1e-16 * sqrt(645000) * 41 = 4e-12
        assert abs(e.virial() - o.virial()) <= 1e-11 * max(abs(o.virial()), abs(o.energy_r())), kernel


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kernel", ["auto", "rows"])
def test_setup_after_charge_change(gpu, precision, kernel):
    """Charges changed after setup hold through a second setup: both ends of a
    pair carry the new ones, as in a fresh engine (the same sums in the same
    order, so the same bits)."""
    print(f"[case] charges over setups {precision} {kernel}", flush=True)
    s = configs.ions(n=600, rho=0.3, kmax=3, seed=5)
    e = Engine(s.copy(), precision=precision)
    e.set_pair_kernel(kernel)
    e.setup()
    e.set_parameters(charge=[0.7, -1.3])
    e.recalculate(force_rebuild=True)
    first = e.get("acc"), e.virial()
    e.setup()
    second = e.get("acc"), e.virial()
    s.charge = np.array([0.7, -1.3])
    f = Engine(s, precision=precision)
    f.set_pair_kernel(kernel)
    f.setup()
    want = f.get("acc"), f.virial()
    for got in (first, second):
        assert np.array_equal(got[0], want[0])
        assert got[1] == want[1]


def test_image_counts_past_a_million_atoms(gpu):
    """More than 4096 workgroups of image counts are scanned by a launch of its
    own: the images bit for bit those of the rule, after the setup, after steps,
    and after a step that failed with others queued behind it."""
    m, box = 102, 76.0                       # 1061208 atoms, at most 40^3 cells
    n = m ** 3
    print(f"[case] scanned image counts n={n}", flush=True)
    g = (np.arange(m) + 0.5) * (box / m)
    pos = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    rng = np.random.default_rng(6)
    pos += rng.uniform(-0.2, 0.2, pos.shape)  # 0.345 apart at least, the LJ reach is 0.2
    s = _free_pair_system(n, box, pos, np.zeros((n, 3)))

    def check(e):
        now = e.get("pos")
        gp, gs = e.ghosts()
        wp, ws = F.numpy_ghosts(s, now)
        assert np.array_equal(gs, ws) and np.array_equal(gp, wp)
        return now

    e = Engine(s)
    e.setup()
    check(e)
    e.set("vel", np.tile([0.5, -0.25, 0.125], (n, 1)))
    e.step(0.125, 3)                          # some atoms wrap
    e.set("vel", np.zeros((n, 3)))
    e.recalculate()
    before = check(e)
    acc = e.get("acc")
    inside = int(np.argmin(((before - box / 2) ** 2).sum(1)))   # an atom without images
    acc[inside] = np.nan
    e.set("acc", acc)
    with pytest.raises(NaNAccelerationError):
        e.step(0.125, 40)
    assert np.array_equal(check(e), before)
    e.set("acc", np.zeros((n, 3)))
    e.step(0.125, 2)
    check(e)


@pytest.mark.parametrize("n", [1048576, 1048577])
def test_kinetic_energy_of_many_workgroups(gpu, n):
    """Up to 4096 workgroups each adds up all sums of m v, past them a launch
    does: kinetic energy, temperature and a Berendsen step of free atoms against
    numpy.  FP64 sums of 1e6 terms of one sign: sqrt(1e6) * 1e-16 = 1e-13."""
    from caviar_amd import BerendsenSettings, ThermoSettings
    print(f"[case] kinetic energy n={n}", flush=True)
    m, box = 102, 102.0
    at = np.arange(n)
    pos = np.stack([at % m, at // m % m, at // (m * m)], axis=1) + 0.5
    rng = np.random.default_rng(n)
    vel = rng.normal(size=(n, 3)) + [0.3, -0.2, 0.1]
    s = _free_pair_system(n, box, np.ascontiguousarray(pos), vel)
    s.mass = np.array([1.5])
    s.thermo = ThermoSettings(k_b=1.1)
    s.berendsen = BerendsenSettings(temperature=0.9, coupling=0.05, dt=0.001)
    e = Engine(s)
    e.setup()
    ke = 0.5 * 1.5 * ((vel - vel.mean(0)) ** 2).sum()
    temp = 2 * ke / (1.1 * (3 * n - 3))
    got = e.thermo()
    assert abs(got[0] - ke) <= 1e-13 * ke and abs(got[1] - temp) <= 1e-13 * temp
    e.step(0.001, 1)
    lam = np.sqrt(1 + 0.001 / 0.05 * (0.9 / temp - 1))
    assert F.rel_err(e.get("vel"), vel * lam) <= 1e-13


def free_bytes():
    """The GPU's free memory (from the HIP runtime the library is linked with)."""
    import ctypes
    from caviar_amd import load_library
    v = [ctypes.c_size_t(), ctypes.c_size_t()]
    assert load_library().hipMemGetInfo(*[ctypes.byref(x) for x in v]) == 0
    return v[0].value


def test_batch_cells_take_room_by_their_own_replica(gpu):
    """A dense replica beside a dilute one of many cells: the batch's memory is
    that of its parts (the dilute one's 140608 cells at 128 bytes a bucket, the
    dense one's rows of about 2100 neighbours), and the pairs are the exact set."""
    print("[case] batch buckets", flush=True)
    rng = np.random.default_rng(4)
    n, box = 5600, 4.5
    dense = _free_pair_system(n, box, rng.uniform(0, box, (n, 3)), np.zeros((n, 3)))
    dilute = _free_pair_system(200, 100.0, rng.uniform(0, 100.0, (200, 3)), np.zeros((200, 3)))
    for s in (dense, dilute):
        s.lj.epsilon[:] = 0.0
    b = Batch([dense, dilute])
    before = free_bytes()
    b.setup()
    used = before - free_bytes()
    assert used <= 300e6, used
    for r, s in enumerate((dense, dilute)):
        gp, _ = F.numpy_ghosts(s, s.pos)
        assert np.array_equal(F.sorted_pairs(b.pairs(r)), F.sorted_pairs(F.exact_pairs(s.pos, gp, 2.0))), r


def test_point_maps_of_many_places(gpu):
    """Maps that take several parts (over 256 MB of phase tables, over 64 MB of
    points and sums): the room they leave behind is bounded, and the values are
    those of the same places asked for in small numbers (FP64: the lattice sums
    of few places are split, 1e-13)."""
    print("[case] point maps", flush=True)
    s = configs.ions(n=300, rho=0.3, kmax=16, seed=3)
    e = Engine(s)
    e.setup()
    rng = np.random.default_rng(2)
    pts = rng.uniform(s.lower, s.upper, (1300007, 3))
    before = free_bytes()
    got = {w: e.point_field(w, pts) for w in ("k", "r")}
    used = before - free_bytes()
    assert used <= 400e6, used
    for at in (0, 200000, 1198372 - 30, 1300007 - 61):
        for w in ("k", "r"):
            f, p = e.point_field(w, pts[at:at + 61])
            assert F.rel_err(got[w][0][at:at + 61], f) <= 1e-13, (w, at)
            assert F.rel_err(got[w][1][at:at + 61], p) <= 1e-13, (w, at)


def test_setup_takes_no_room_for_the_adjoint(gpu):
    """What only the adjoint uses is taken at its first call, once: a setup of
    8000 ions leaves less than 50 MB, the adjoint's partial sums come to 20."""
    print("[case] setup room", flush=True)
    s = configs.ions(n=8000, rho=0.3, kmax=8, seed=3)
    e = Engine(s)
    before = free_bytes()
    e.setup()
    at_setup = free_bytes()
    w = np.random.default_rng(1).normal(size=(s.n, 3))
    g = e.adjoint(w)
    first = free_bytes()
    for _ in range(3):
        assert np.array_equal(e.adjoint(w)[2], g[2])
    assert free_bytes() == first
    assert before - at_setup <= 50e6, before - at_setup
    assert np.array_equal(e.adjoint_noalloc(w)[2], g[2])
    f = Engine(s)              # the scratch's adjoint without the room: the same bits
    f.setup()
    assert np.array_equal(f.adjoint_noalloc(w)[2], g[2])
