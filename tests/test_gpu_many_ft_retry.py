"""Force and torque of many solids, handed over beside the field pass, where a step does not succeed
the first time (needs an MI355X): a step that fails in the end, and steps run again with larger
buffers or other tile classes, big tiles among them.  Every row as where nothing had to be repeated,
bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from sdfibm_amd import _lib
from sdfibm_amd import mesh as M
from sdfibm_amd import solids as S
from sdfibm_amd.cloud import SolidCloud

pytestmark = pytest.mark.gpu

DT = 1e-3


def _cloud(mesh, seed):
    c = SolidCloud(mesh, rho_f=1.0, precision="fp32")
    c.set_velocity(np.random.default_rng(seed).normal(0, 1.0, (mesh.n_cells, 3)))
    return c


def _grid(n, step, margin):
    g = np.stack(np.meshgrid(*(np.arange(k) for k in n), indexing="ij"), -1).reshape(-1, 3)
    return g * np.array(step) + margin


def test_a_failed_step_hands_over_its_rows():
    """140 solids over one brick among 16,700: ERR_CAPACITY, and the rows of both halves alone."""
    e = 84
    mesh = M.uniform_box((e, e, e), (0, 0, 0), (float(e),) * 3)
    rng = np.random.default_rng(11)
    at = _grid((26, 26, 26), (3.0,) * 3, 5.5)[:16560]
    sol = S.make_solids(140 + len(at))
    sol["shape"] = S.SPHERE
    sol["prm"][:, 0] = rng.uniform(0.9, 1.2, sol.size)
    sol["center"] = np.concatenate([np.full((140, 3), 1.9), at + rng.uniform(-0.2, 0.2, at.shape)])
    sol["center"][:140] += rng.uniform(-0.3, 0.3, (140, 3))
    sol["vel"] = rng.normal(0, 0.1, (sol.size, 3))
    half = [np.r_[0:70, 140:9000], np.r_[70:140, 9000:sol.size]]
    with _cloud(mesh, 1) as c:
        c.set_solids(sol)
        ft = np.full((sol.size, 6), np.nan)
        assert _lib.load().sdfibm_interact(c._h, 0.0, DT, ft.ctypes.data) == -8
        for h in half:
            c.set_solids(sol[h])
            np.testing.assert_array_equal(ft[h], c.interact(0.0, DT))


@pytest.mark.parametrize("what", ["grown", "oversized"])
def test_steps_run_again(what):
    """grown: slender ellipsoids turned to the diagonal through set_solids' fast path, their tiles three
    times as large as the code buffer allows for.  oversized: a rod turned to the diagonal, its
    tile beyond the big-tile pass."""
    rng = np.random.default_rng(12)
    if what == "grown":
        mesh = M.uniform_box((168, 112, 112), (0, 0, 0), (168.0, 112.0, 112.0))
        at = _grid((27, 25, 25), (6.0, 4.0, 4.0), 5.0)
    else:
        mesh = M.uniform_box((300, 160, 160), (0, 0, 0), (300.0, 160.0, 160.0))
        at = _grid((40, 22, 20), (7.0, 7.0, 7.5), 6.0)
    sol = S.make_solids(len(at) + 2)
    assert sol.size >= 16384
    sol["center"][2:] = at + rng.uniform(-0.2, 0.2, at.shape)
    sol["center"][:2] = np.array([mesh.nx, mesh.ny, mesh.nz]) * [[0.5, 0.5, 0.5], [0.3, 0.6, 0.4]]
    sol["vel"] = rng.normal(0, 0.1, (sol.size, 3))
    turned = sol["center"].copy()
    q = S.quaternion_xyz((0.0, -np.arctan(1 / np.sqrt(2.0)), np.pi / 4))
    if what == "grown":
        sol["shape"] = S.ELLIPSOID
        sol["prm"][:, :3] = 4.0, 0.6, 0.6
        sol["prm"][:2, :3] = 35.0, 10.0, 9.0  # big tiles
    else:
        sol["shape"] = S.SPHERE
        sol["prm"][:, 0] = 1.2
        sol["shape"][:2] = S.BOX
        sol["prm"][:2, :3] = [(170.0, 2.0, 2.0), (36.0, 9.0, 8.0)]
    later = sol.copy()
    later["center"] = turned
    later["q"] = q
    with _cloud(mesh, 2) as c:
        c.set_solids(sol)
        first = c.interact(0.0, DT)
        cap = c.buffer_capacity()
        c.set_solids(later)
        ft = c.interact(0.0, DT)
        if what == "grown":
            assert c.buffer_capacity()[0] > cap[0]  # the step ran again
        with _cloud(mesh, 2) as f:
            f.set_solids(later)
            np.testing.assert_array_equal(ft, f.interact(0.0, DT))
    assert np.any(ft != first, axis=1)[:2].all()
