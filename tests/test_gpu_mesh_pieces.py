"""GPU: cell areas whose integrals are split at the regions' breaks, where the
split can go wrong: circles through the pole and nearly so, thin rings, a cut
circle across the region's edge or touching it from inside, and the smallest
mesh, against the oracle's adaptive integrals (xpsi/cellmesh/mesh.pyx:23-417,
polar_mesh.pyx:23-430, mesh_tools.pyx:429-725)."""
import math

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

# name, radius, colatitude, cut radius, cut colatitude, cut azimuth, cells a side
CASES = [
    ("spot-2", 0.3, 1.1, 0.0, 1.1, 0.0, 2),
    ("thin-ring", 0.31, 0.9, 0.3, 0.9, 0.0, 20),
    ("cut-across-edge", 0.3, 1.2, 0.2, 1.35, 0.2, 16),
    ("cut-touches-inside", 0.3, 1.2, 0.1, 1.4, 0.0, 16),
    ("near-pole", 0.4, 0.4001, 0.0, 0.4001, 0.0, 14),
    ("over-pole", 0.4001, 0.4, 0.0, 0.4, 0.0, 14),
    ("cut-over-pole", 0.5, 0.3, 0.31, 0.3, 0.0, 18),
    ("south-cut-offset", 0.5, math.pi - 0.2, 0.2, math.pi - 0.3, 0.4, 18),
]


@pytest.fixture(scope="module")
def star():
    return O.spacetime(1.4, 12.0, 1.0, 0.5, 300.0, "AGM_14")


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_cell_areas_at_breaks(star, case):
    from xpsi_amd.cellmesh.mesh import construct_polar_cellMesh, construct_spot_cellMesh
    _, rad, col, cut, ccol, cazi, S = case
    st = star
    polar = (col - rad < 0.0) or (col + rad > math.pi)
    args = (S * S, S, st["M"], st["r_s"], st["R"], st["zeta"], st["epsilon"], st["shape"], rad, col, cut, ccol, cazi)
    fn = construct_polar_cellMesh if polar else construct_spot_cellMesh
    got = fn(1, *args)[3]
    ref = O.construct_cell_mesh(polar, *args)[3]
    # the reference's integrals are adaptive to 1e-10 of themselves, each over
    # the cell or up to four pieces of it; positions are rounded to 1e-16 of a
    # radian, some 1e-13 of a cell's extent
    assert np.all(np.abs(got - ref) <= 4e-10 * np.abs(ref) + 1e-12 * ref.max())
    assert np.array_equal(got > 0.0, ref > 0.0)
