"""What the voxelizer's classification leaves to the tests, for faces in voxel planes and for
triangles without an area: the answers are the tests' (as in test_walk_bounds), and most columns
are decided without them."""
import numpy as np
import pytest

from test_walk_bounds import check  # noqa: F401  (the fixture)

_FACES = [(0, 1, 3), (0, 3, 2), (4, 6, 7), (4, 7, 5), (0, 4, 5), (0, 5, 1), (2, 3, 7), (2, 7, 6),
          (0, 2, 6), (0, 6, 4), (1, 5, 7), (1, 7, 3)]


def boxes(rng, n, lo, hi, G):
    """n boxes of lo to hi voxels a side with their corners on voxel corners."""
    size = np.round(rng.uniform(lo, hi, (n, 1, 3)))
    at = np.round(rng.uniform(1, G - 1 - hi, (n, 1, 3)))
    corner = np.array([[x, y, z] for x in (0, 1) for y in (0, 1) for z in (0, 1)], float)[None]
    return ((at + corner * size) / G)[:, np.array(_FACES)].reshape(-1, 9).astype(np.float32)


def without_area(rng, n, size, G):
    """Three points on a line, on fractions of a voxel that are exact."""
    a = np.round(rng.uniform(0.1, 0.9, (n, 3)) * 8 * G) / (8 * G)
    d = np.round(rng.normal(size=(n, 3)) * size * 8) / (8 * G)
    return np.stack([a, a + d, a + 2 * d], 1).reshape(n, 9).astype(np.float32)


@pytest.mark.parametrize("unit", [1.0, 0.77777779])
@pytest.mark.parametrize("G", [64, 1024, 32768])
def test_faces_in_voxel_planes(check, G, unit):  # noqa: F811
    tris = boxes(np.random.default_rng(G), 150, 4, 30, G)
    got = check(tris * np.float32(unit), G, unit=unit / G)
    assert got["wrong"] == 0 and got["accepted"] > 0, got
    assert got["uncertain"] < 0.25 * got["columns"], got  # rows' ends, edges


@pytest.mark.parametrize("G", [64, 1024])
def test_faces_a_hair_off_voxel_planes(check, G):  # noqa: F811
    """A few units in the last place away: still decided by the tests' own rounding."""
    rng = np.random.default_rng(G)
    tris = boxes(rng, 100, 2, 12, G)
    tris += (rng.integers(-3, 4, (len(tris), 1)) * np.spacing(tris)).astype(np.float32)
    got = check(tris, G)
    assert got["wrong"] == 0 and got["accepted"] > 0, got


@pytest.mark.parametrize("G", [64, 1024])
def test_triangles_without_area(check, G):  # noqa: F811
    """Only the columns of a row's interval go through the tests, not all of the bbox."""
    tris = without_area(np.random.default_rng(G), 400, 4.0, G)
    got = check(tris, G)
    assert got["wrong"] == 0 and got["accepted"] > 0, got
    g = np.floor(tris.reshape(-1, 3, 3).astype(np.float64) * G)
    side = np.sort(g.max(1) - g.min(1) + 1, axis=1)
    assert got["columns"] < 0.6 * (side[:, 1] * side[:, 0]).sum(), (got, side.shape)
