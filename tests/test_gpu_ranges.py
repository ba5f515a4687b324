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
