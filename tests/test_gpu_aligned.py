"""Faces in voxel planes, faces a hair off them and triangles without an area, against the oracle."""
import numpy as np
import pytest

import oracle
from ooc_svo_builder_amd import SvoContext
from test_walk_aligned import boxes, without_area

pytestmark = pytest.mark.gpu
G = 128


def _mesh(kind, payload):
    rng = np.random.default_rng(21)
    if kind == "area":
        geo = np.concatenate([without_area(rng, 300, s, G) for s in (1.0, 8.0)])
    else:
        geo = np.concatenate([boxes(rng, 60, 2, 8, G), boxes(rng, 12, 20, 60, G)])
        if kind == "hair":
            geo += (rng.integers(-3, 4, (len(geo), 1)) * np.spacing(geo)).astype(np.float32)
    geo = geo[rng.permutation(len(geo))]
    return np.concatenate([geo, rng.uniform(0, 1, (len(geo), 12)).astype(np.float32)], 1) if payload else geo


@pytest.fixture(scope="module")
def want():
    return {(k, p): oracle.pipeline(_mesh(k, p), p, G, 2048) for k in ("plane", "hair", "area")
            for p in (False, True)}


@pytest.mark.parametrize("small_cols,direct", [(1024, 16), (1024, 0), (1, 0), (100, 0)])
@pytest.mark.parametrize("dense", [True, False])
@pytest.mark.parametrize("payload", [False, True])
@pytest.mark.parametrize("kind", ["plane", "hair", "area"])
def test_aligned_meshes(kind, payload, dense, small_cols, direct, want):
    tris = _mesh(kind, payload)
    nodes, data, hz, _, nf = want[kind, payload]
    with SvoContext(0) as ctx:
        ctx.set_tuning(dense_limit_mb=None if dense else 0)
        k = ctx.get_tuning()
        ctx.set_knobs(small_cols, direct, k[2], k[3])
        info = ctx.run(tris, payload, G)
        assert (info.nfilled, info.hazard) == (nf, hz)
        assert ctx.nodes(info.n_nodes).tobytes() == nodes.tobytes()
        assert ctx.data(info.n_data).tobytes() == data.tobytes()
