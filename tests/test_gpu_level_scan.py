"""The generic build without -levels around the size where its level scans change."""
import numpy as np
import pytest

import oracle
from ooc_svo_builder_amd import SvoContext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("levels", [False, True])
@pytest.mark.parametrize("n", [(1 << 21) - 1, 1 << 21, (1 << 21) + 1])
def test_voxel_counts_around_two_million(n, levels):
    G = 256
    codes = np.sort(np.random.default_rng(n).permutation(G ** 3)[:n]).astype(np.uint64)
    nodes, data = oracle.build_octree(codes, G, False, levels)[:2]
    with SvoContext(0) as ctx:
        ctx.load_mesh(np.zeros((0, 9), np.float32), False)
        ctx.add_voxels(codes)
        nn, nd, _ = ctx.build(G, levels)
        assert (nn, nd) == (len(nodes), len(data))
        assert ctx.nodes(nn).tobytes() == nodes.tobytes()
        assert ctx.data(nd).tobytes() == data.tobytes()
