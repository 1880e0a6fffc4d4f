"""Passes on touched bricks that find more of them than there are slots, against the oracle."""
import numpy as np
import pytest

import oracle
from ooc_svo_builder_amd import SvoContext

pytestmark = pytest.mark.gpu


def _mesh(rng, n, G, payload):
    c = rng.uniform(0.02, 0.98, (n, 1, 3))
    geo = (c + rng.normal(size=(n, 3, 3)) * 1.5 / G).reshape(n, 9).astype(np.float32)
    return np.concatenate([geo, rng.uniform(0, 1, (n, 12)).astype(np.float32)], 1) if payload else geo


@pytest.mark.parametrize("payload", [False, True])
def test_more_bricks_than_slots(payload):
    """1,024 slots at first; one context over meshes of ~900, 9,000, 30,000 and 9,000 bricks."""
    G = 512
    rng = np.random.default_rng(12)
    with SvoContext(0) as ctx:
        ctx.set_tuning(dense_limit_mb=0)
        for n in (600, 7000, 60000, 7000):
            print("touched bricks of %d triangles" % n, flush=True)
            tris = _mesh(rng, n, G, payload)
            nodes, data, hz, _, nf = oracle.pipeline(tris, payload, G, 2048)
            info = ctx.run(tris, payload, G)
            assert (info.nfilled, info.hazard) == (nf, hz)
            assert ctx.nodes(info.n_nodes).tobytes() == nodes.tobytes()
            assert ctx.data(info.n_data).tobytes() == data.tobytes()
