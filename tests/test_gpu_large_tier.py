"""The column-parallel tier's lists at and past their ends, against the oracle: set-ups that are
not stored, jobs that find no place and are dealt to all waves, triangles left to one wave."""
import numpy as np
import pytest

import oracle
from ooc_svo_builder_amd import SvoContext

pytestmark = pytest.mark.gpu


def _mesh(payload):
    """Triangles over most of the grid (one row a job, or a few), of about ten rows a job and of
    fewer columns than a wave, and some of the small tier."""
    rng = np.random.default_rng(11)
    tris = []
    for n, size in ((6, 0.9), (12, 0.4), (40, 0.12), (60, 0.01)):
        c = rng.uniform(size / 2, 1 - size / 2, (n, 1, 3))
        tris.append((c + rng.uniform(-size / 2, size / 2, (n, 3, 3))).reshape(n, 9))
    tris = np.concatenate(tris)[rng.permutation(118)].astype(np.float32)
    return np.concatenate([tris, rng.uniform(0, 1, (118, 12)).astype(np.float32)], 1) if payload else tris


@pytest.mark.parametrize("small_cols", [64, 1])
@pytest.mark.parametrize("payload", [False, True])
def test_triangles_of_few_and_many_jobs(payload, small_cols):
    """Tiles whose lanes have no further job, up to 8 (written by the lane) and more (by the wave)."""
    G, tris = 256, _mesh(payload)
    with SvoContext(0) as ctx:
        ctx.set_tuning(small_cols=small_cols)
        for limit in (2048, 2):
            nodes, data, _, parts, nf = oracle.pipeline(tris, payload, G, limit)
            info = ctx.run(tris, payload, G, limit)
            assert (info.n_partitions, info.nfilled) == (parts, nf)
            assert ctx.nodes(info.n_nodes).tobytes() == nodes.tobytes()
            assert ctx.data(info.n_data).tobytes() == data.tobytes()


@pytest.fixture(scope="module")
def want():
    G = 256
    return {p: (oracle.pipeline(_mesh(p), p, G, 2048), oracle.pipeline(_mesh(p), p, G, 2)) for p in (False, True)}


@pytest.mark.parametrize("room", [(1 << 16, 1 << 20), (0, 0), (3, 0), (1 << 16, 0), (1 << 16, 1), (5, 100),
                                  (0, 300), (20, 400)])
@pytest.mark.parametrize("dense", [True, False])
@pytest.mark.parametrize("payload", [False, True])
def test_lists_past_their_room(payload, dense, room, want):
    """small_cols 64 and 1: the larger kinds of triangles in jobs, and all of them; one partition
    and eight. What the lists have no room for gives the same bytes."""
    G, tris = 256, _mesh(payload)
    with SvoContext(0) as ctx:
        ctx.set_tuning(dense_limit_mb=None if dense else 0)
        ctx.set_large_tier(*room)
        k = ctx.get_tuning()
        for small_cols in (64, 1):
            for blocks in (k[3], 2):
                ctx.set_knobs(small_cols, 0, k[2], blocks)
                for (nodes, data, _, parts, nf), limit in zip(want[payload], (2048, 2)):
                    info = ctx.run(tris, payload, G, limit)
                    assert (info.n_partitions, info.nfilled) == (parts, nf)
                    assert ctx.nodes(info.n_nodes).tobytes() == nodes.tobytes()
                    assert ctx.data(info.n_data).tobytes() == data.tobytes()
