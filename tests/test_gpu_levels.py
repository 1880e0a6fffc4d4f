"""The generic build (voxels from outside, -levels) around the sizes where its passes change."""
import numpy as np
import pytest

import oracle
from ooc_svo_builder_amd import SvoContext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,G,levels", [(4095, 64, True), (4097, 64, True), (70000, 64, True),
                                       (8193, 32768, True), (65537, 32768, False),
                                       ((1 << 23) - 1, 256, False), ((1 << 23) + 1, 256, True)])
def test_voxel_counts_around_the_pass_sizes(n, G, levels):
    """Level scans of one element a thread and of eight, the small levels' one-block passes,
    with and without -levels, against the oracle's octree."""
    rng = np.random.default_rng(n)
    if n > G ** 3 // 4:
        codes = np.sort(rng.permutation(G ** 3)[:n]).astype(np.uint64)
    else:
        codes = np.unique(rng.integers(0, G ** 3, 2 * n, dtype=np.uint64))
        codes = np.sort(rng.choice(codes, n, replace=False))
    want_nodes, want_data, _ = oracle.build_octree(codes, G, False, levels)[:3]
    with SvoContext(0) as ctx:
        ctx.load_mesh(np.zeros((0, 9), np.float32), False)
        ctx.add_voxels(codes)
        nn, nd, _ = ctx.build(G, levels)
        assert (nn, nd) == (len(want_nodes), len(want_data))
        assert ctx.nodes(nn).tobytes() == want_nodes.tobytes()
        assert ctx.data(nd).tobytes() == want_data.tobytes()
