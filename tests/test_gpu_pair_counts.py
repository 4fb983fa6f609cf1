"""pair_counts is the sum of the solids' candidate lists where some solids have left the mesh (needs an
MI355X): a solid without a tile counts nothing, whatever its last counts were."""
from __future__ import annotations

import numpy as np
import pytest

from sdfibm_amd import mesh as M
from sdfibm_amd import solids as S
from sdfibm_amd.cloud import SolidCloud

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["rect", "struct", "poly"])
def test_solids_outside_the_mesh(kind):
    mesh = M.uniform_box((24, 20, 16), (0, 0, 0), (24.0, 20.0, 16.0))
    sol = S.make_solids(6)
    sol["prm"][:, 0] = 2.5
    sol["center"] = [(5, 5, 5), (12, 10, 8), (18, 6, 9), (6, 14, 10), (17, 14, 4), (12, 4.3, 8)]
    sol["shape"][5], sol["prm"][5] = S.PLANE, 0
    with SolidCloud(mesh.to_polymesh() if kind == "poly" else mesh, precision="fp32",
                    force_structured=kind == "struct") as c:
        for gone in ([], [1, 4], [0], []):
            now = sol.copy()
            now["center"][gone] += 100.0
            c.set_solids(now)
            c.interact(0.0, 1e-3)
            lists = np.sum([c.candidates(s)[0][:3] for s in range(6)], axis=0)
            assert c.pair_counts() == (lists[0], lists[1] + lists[2])
