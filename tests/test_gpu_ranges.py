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
from caviar_amd import Engine, configs
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
