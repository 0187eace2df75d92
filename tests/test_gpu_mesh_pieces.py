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


SMALL = [(0.0251, 0.3784, 0.0, 0.3784, 0.0, 128), (0.0516, 0.1695, 0.0227, 0.166, -0.0008, 128),
         (0.0247, 1.1896, 0.0057, 1.1896, 0.0, 96)]


@pytest.mark.parametrize("case", SMALL, ids=["spot", "cut-off-centre", "cut"])
def test_small_spots(star, case):
    """Spots whose slivers cannot be known to 1e-12 of themselves."""
    from xpsi_amd.cellmesh.mesh import construct_spot_cellMesh
    rad, col, cut, ccol, cazi, S = case
    st = star
    args = (S * S, S, st["M"], st["r_s"], st["R"], st["zeta"], st["epsilon"], st["shape"], rad, col, cut, ccol, cazi)
    got, ref = construct_spot_cellMesh(1, *args)[3], O.construct_cell_mesh(False, *args)[3]
    # as above, and the circles' azimuths: acos of (cos R - cos C cos t) / (sin C
    # sin t), off by an ulp or two before the acos, so by that over R sin C behind
    # it, against a cell's 2 R / (S sin C); on both sides
    r = cut if cut else rad
    noise = 4 * S * np.finfo(float).eps / r ** 2
    assert np.all(np.abs(got - ref) <= 4e-10 * np.abs(ref) + noise * ref.max())
    assert np.array_equal(got > noise * ref.max(), ref > noise * ref.max())


def test_small_spots_take_no_longer(star):
    """Small spots' boundary cells are as many as a large one's and settle as soon
    (with their slivers bisected in vain these meshes took up to three times
    as long)."""
    import time
    from xpsi_amd.cellmesh.mesh import construct_spot_cellMesh
    st, S = star, 256
    best = {}
    for _ in range(6):
        for rad in (0.3, 0.02, 0.025, 0.03, 0.04, 0.05):
            args = (S * S, S, st["M"], st["r_s"], st["R"], st["zeta"], st["epsilon"], st["shape"], rad, 0.3784, 0.0,
                    0.3784, 0.0)
            t = time.perf_counter()
            construct_spot_cellMesh(1, *args)
            best[rad] = min(best.get(rad, 1.0), time.perf_counter() - t)
    print("[gpu] mesh of 256 x 256: " + ", ".join("radius %.3f %.0f us" % (r, t * 1e6) for r, t in best.items()), flush=True)
    assert max(best.values()) < 1.5 * best[0.3]
