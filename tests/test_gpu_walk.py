"""The voxelizer's wave-wide walks at the edges of their tiles and jobs, against the oracle."""
import numpy as np
import pytest

import oracle
from ooc_svo_builder_amd import SvoContext

pytestmark = pytest.mark.gpu


def _codes(ctx, tris, payload, G):
    ctx.load_mesh(tris, payload)
    ctx.voxelize(0, 0, G ** 3, 1.0 / G, G)
    return ctx.codes()


def _want(tris, payload, G):
    codes, _ = oracle.voxelize(tris, payload, 0, G ** 3, 1.0 / G)
    return np.sort(codes)


def _mesh(rng, n, size):
    c = rng.uniform(0.1, 0.9, (n, 1, 3))
    return (c + rng.normal(size=(n, 3, 3)) * size).reshape(n, 9).astype(np.float32)


@pytest.mark.parametrize("direct", [0, 16])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 16 * 4096 + 1])
def test_tile_edges(n, direct):
    """Triangle counts around a wave's 64 and around one tile per wave."""
    G = 128
    tris = _mesh(np.random.default_rng(n), n, 2.0 / G if n > 1000 else 6.0 / G)
    with SvoContext(0) as ctx:
        k = ctx.get_tuning()
        ctx.set_knobs(k[0], direct, k[2], k[3])
        assert np.array_equal(_codes(ctx, tris, False, G), _want(tris, False, G))


@pytest.mark.parametrize("small_cols", [4, 1024, 1 << 20])
@pytest.mark.parametrize("aligned", [False, True])
def test_large_triangles_in_jobs(small_cols, aligned):
    """Triangles of up to 256 x 256 columns: jobs of a few rows each, rows of more columns than
    a wave, and faces on voxel planes, whose columns all go through the tests."""
    G = 256
    rng = np.random.default_rng(5)
    tris = rng.uniform(0.0, 1.0, (9, 9)).astype(np.float32)
    if aligned:
        tris = (np.round(tris * 16) / 16).astype(np.float32)
        tris[:, 2] = tris[:, 5] = tris[:, 8]
    with SvoContext(0) as ctx:
        ctx.set_tuning(small_cols=small_cols)
        assert np.array_equal(_codes(ctx, tris, False, G), _want(tris, False, G))


def test_bbox_ends_beyond_int():
    """A coordinate past the range of int truncates to INT_MIN as on x86: its bbox is inverted
    or clamped to the grid's first layer."""
    G = 64
    tris = _mesh(np.random.default_rng(8), 300, 3.0 / G)
    tris[::5, 3] = 1e12
    tris[1::5, 7] = -1e12
    tris[2::5, 2] = 3e38
    with SvoContext(0) as ctx:
        assert np.array_equal(_codes(ctx, tris, False, G), _want(tris, False, G))


@pytest.mark.parametrize("size", [1.0, 40.0])
def test_words_and_flags_are_clear_again(size):
    """The same context over another mesh and back: no mark, flag or cell is left behind."""
    G = 128
    rng = np.random.default_rng(3)
    a, b = _mesh(rng, 500, size / G), _mesh(rng, 700, 2.0 / G)
    pay = np.concatenate([b, rng.uniform(0, 1, (700, 12)).astype(np.float32)], axis=1)
    with SvoContext(0) as ctx:
        want = _want(a, False, G)
        for mesh, payload in ((a, False), (pay, True), (b, False), (a, False)):
            got = _codes(ctx, mesh, payload, G)
            if mesh is a:
                assert np.array_equal(got, want)
            else:
                assert np.array_equal(got, _want(mesh, payload, G))


def test_fresh_context_waits_for_its_own_read_back():
    """A new context's pinned read-back area may be memory a closed context left its completion
    flag in: the first read-back must not take that flag for its own."""
    G = 128
    for n in (1, 40, 200):
        tris = _mesh(np.random.default_rng(n), n, 6.0 / G)
        with SvoContext(0) as ctx:
            assert np.array_equal(_codes(ctx, tris, False, G), _want(tris, False, G))
