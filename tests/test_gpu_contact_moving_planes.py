"""evolve with contacts among planes that move and turn, against the oracle (needs an MI355X): every
sub-step takes the planes as the sub-step before left them, in the one-workgroup form and beyond its
1,024 solids.  Same formulas in another order of loads: 1e-12 of the largest value."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from sdfibm_amd import mesh as M
from sdfibm_amd import solids as S
from sdfibm_amd.cloud import SolidCloud

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 200, 900, 1100])
def test_moving_planes(n):
    rng = np.random.default_rng(n)
    e = 48
    mesh = M.uniform_box((e, e, e), (0, 0, 0), (float(e),) * 3)
    sol = S.make_solids(n + 3)
    sol["prm"][:n, 0] = rng.uniform(1.0, 1.9, n)
    at = rng.permutation(12 ** 3)[:n]
    sol["center"][:n] = np.stack([at % 12, at // 12 % 12, at // 144], 1) * 3.9 + 2.5 + rng.uniform(-0.3, 0.3, (n, 3))
    sol["shape"][n:] = S.PLANE
    sol["center"][n:] = [(24, 9, 24), (8, 24, 24), (24, 24, 40)]
    for t, q in enumerate([(0.1, 0, 0.2), (0.0, 0.3, -1.5), (-1.6, 0.1, 0.0)]):
        sol["q"][n + t] = S.quaternion_xyz(q)
    sol["vel"] = rng.normal(0, 5.0, (n + 3, 3))
    sol["omega"] = rng.normal(0, 2.0, (n + 3, 3))
    with SolidCloud(mesh, rho_f=1.0, precision="fp64") as c:
        c.set_solids(sol)
        c.set_dynamics(2.0)
        c.set_contact(2000.0, 1.0)
        c.evolve(0.0, 0.02, (0.0, -1.0, 0.0))
        got = c.solids()
    dyn = oracle.make_dyn(n + 3, 2.0)
    ref, _ = oracle.evolve_contact(sol, dyn, np.zeros((n + 3, 6)), 0.0, 0.02, (0.0, -1.0, 0.0), 1.0, 2000.0, 1.0)
    for k in ("center", "q", "vel", "omega"):
        scale = np.abs(ref[k]).max()
        assert np.max(np.abs(got[k] - ref[k])) <= 1e-12 * scale, k
    assert np.abs(ref["vel"] - sol["vel"]).max() > 0.1  # the contacts acted
