"""Solids whose first-order distance is infinite at a mesh vertex, against the oracle (needs an
MI355X): an ellipsoid's distance is -inf at its centre, and +inf where the ellipsoid is taken off.
Centres on vertices inside the mesh and on its faces, edges and corners; the cell size is a power of
two and the solids are not rotated, so the distance there is infinite in both precisions.  A cell
whose fraction the formulas give finite has that fraction; one they give none for is not listed.
Tolerances of test_gpu_parity.py."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from _helpers import split_candidates
from sdfibm_amd import mesh as M
from sdfibm_amd import solids as S
from sdfibm_amd.cloud import SolidCloud

pytestmark = pytest.mark.gpu

H = 1.0 / 8
TOL = {"fp64": 1e-12, "fp32": 1e-6}


def _scene(shape, size, flat=False, jitter=0.0):
    """One solid of `size` cells (a shape id, or CSG primitives in units of `size`) on each of some
    vertices of a 24 x 20 x 16 (x 1) mesh: mesh, solids, CSG table."""
    n = (24, 20, 1) if flat else (24, 20, 16)
    box = (0, 0, -0.5 if flat else 0), (n[0] * H, n[1] * H, 0.5 if flat else n[2] * H)
    mesh = M.jittered_box(n, *box, jitter, 3) if jitter else M.uniform_box(n, *box)
    g = np.meshgrid((0, 6, 12, 18, 24), (0, 7, 13, 20), (0,) if flat else (0, 8, 16), indexing="ij")
    at = np.stack(g, -1).reshape(-1, 3)
    sol = S.make_solids(len(at))
    sol["center"] = np.asarray(mesh.points)[at[:, 0] + (n[0] + 1) * (at[:, 1] + (n[1] + 1) * at[:, 2])]
    if flat:
        sol["center"][:, 2] = 0.0
    table = None
    if isinstance(shape, int):
        sol["shape"] = shape
        sol["prm"][:, :3] = np.array([1.0, 0.85, 0.95 if shape == S.ELLIPSOID else 0.0]) * size * H
    else:
        sol["shape"] = S.CSG
        table = S.csg_shape([dict(kind=k, op=op, size=np.array(s) * size * H) for k, op, s in shape], volume=1.0,
                            moi=(1.0, 1.0, 1.0), radius_b=3.0 * size * H)
    sol["vel"] = np.random.default_rng(5).normal(0, 0.1, (sol.size, 3))
    return mesh, sol, table


def _lists(mesh, sol, table, prec, flat=False, structured=False):
    with SolidCloud(mesh, two_d=flat, rho_f=1.0, precision=prec, force_structured=structured) as c:
        if table is not None:
            c.set_csg_shapes(table)
        c.set_solids(sol)
        c.set_velocity(np.ones((mesh.n_cells, 3)))
        c.interact(0.0, 1e-3)
        return [c.candidates(s)[1:] for s in range(sol.size)]


def _against_oracle(mesh, sol, table, prec, flat=False, poly=False, structured=False):
    pm = mesh.to_polymesh()
    if table is not None:
        oracle.set_csg(np.atleast_1d(table))
    r = oracle.OracleMesh(pm).interact(sol, np.ones((mesh.n_cells, 3)), two_d=flat, rho_f=1.0, dt=1e-3,
                                       capture=True, capacity=40 * mesh.n_cells)
    got = _lists(pm if poly else mesh, sol, table, prec, flat, structured)
    worst = 0.0
    for s, (_, cells, alpha) in enumerate(split_candidates(r, sol.size)):
        ref = {int(c): a for c, a in zip(cells, alpha) if np.isfinite(a)}
        have = dict(zip((int(c) for c in got[s][0]), got[s][1]))
        assert set(have) == set(ref), (s, sorted(set(have) ^ set(ref)))
        worst = max([worst] + [abs(have[c] - ref[c]) for c in ref])
    assert worst <= TOL[prec]


VOID = [("box", "union", (1.3, 1.3, 1.3)), ("ellipsoid", "difference", (0.6, 0.6, 0.6))]


@pytest.mark.parametrize("size", [0.6, 0.95, 1.2, 1.7])
@pytest.mark.parametrize("poly", [False, True])
def test_ellipsoid_taken_off(poly, size):
    """A finite distance over the infinite one of the void's centre is 0."""
    _against_oracle(*_scene(VOID, size), "fp64", poly=poly)


@pytest.mark.parametrize("size", [0.6, 0.95, 1.2, 1.7])
def test_ellipsoid_taken_off_structured(size):
    """The general hexahedron's two precisions list the same cells."""
    mesh, sol, table = _scene(VOID, size)
    a, b = (_lists(mesh, sol, table, prec, structured=True) for prec in ("fp64", "fp32"))
    for (ca, fa), (cb, fb) in zip(a, b):
        np.testing.assert_array_equal(ca, cb)
        assert np.max(np.abs(fa - fb), initial=0.0) <= TOL["fp32"]


BALL = [("ellipsoid", "union", (1.0, 0.9, 1.1))]
FLAT_VOIDS = ([("box", "union", (1.3, 1.3, 1.3)), ("ellipsoid", "difference", (0.35, 1.25, 1.2))],
              [("sphere", "union", (1.5,)), ("ellipsoid", "difference", (1.25, 0.35, 1.2))],
              [("sphere", "union", (1.5,)), ("ellipsoid", "difference", (1.25, 1.2, 0.35))])


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("size", [0.6, 0.95, 1.2, 1.45, 1.7, 2.3])
@pytest.mark.parametrize("which", ["ellipse2d", "ellipse3d", "csg"])
def test_centre_on_a_vertex(which, size, prec):
    """A cut cell with a corner at -inf: its edges to inside corners lie inside."""
    flat = which == "ellipse2d"
    _against_oracle(*_scene(BALL if which == "csg" else S.ELLIPSE, size, flat), prec, flat)


@pytest.mark.parametrize("size", [0.6, 0.95, 1.2])
def test_ellipsoid_centre_on_a_vertex_fp32(size):
    _against_oracle(*_scene(S.ELLIPSOID, size), "fp32")


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("size", [0.6, 0.8, 0.95, 1.2, 1.7])
@pytest.mark.parametrize("void", range(len(FLAT_VOIDS)))
def test_faces_outside_with_a_corner_at_infinity(void, size, prec):
    """A face of a cut cell wholly outside whose first corner is the void's centre has no area inside."""
    _against_oracle(*_scene(FLAT_VOIDS[void], size), prec)


@pytest.mark.parametrize("axes", [(0.6, 1.5, 1.6), (1.5, 0.6, 1.6), (1.6, 1.5, 0.6), (0.9, 0.8, 2.2), (1.2, 1.1, 1.0)])
def test_ellipsoid_centre_on_a_vertex_fp64(axes):
    """The reciprocal root of the zero squared length at the centre is infinite, not NaN: an edge from
    there to outside has no fraction."""
    mesh, sol, _ = _scene(S.ELLIPSOID, 1.0)
    sol["prm"][:, :3] = np.array(axes) * H
    _against_oracle(mesh, sol, None, "fp64")


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("jitter", [0.0, 0.15])
@pytest.mark.parametrize("size", [0.6, 0.95, 1.2, 1.7])
@pytest.mark.parametrize("which", ["ellipse2d", "ellipsoid", "csg", "void0", "void1", "void2"])
def test_general_hexahedra(which, size, jitter, prec):
    """Cells of eight points that are not boxes: the corners the cell's apex does not take have no weight."""
    flat = which == "ellipse2d"
    shape = FLAT_VOIDS[int(which[-1])] if which.startswith("void") else \
        dict(ellipse2d=S.ELLIPSE, ellipsoid=S.ELLIPSOID, csg=BALL)[which]
    _against_oracle(*_scene(shape, size, flat, 0.0 if flat else jitter), prec, flat, structured=True)
