"""The stages' times that a run reports (svo_run_info)."""
import time

import pytest

from ooc_svo_builder_amd import SvoContext, generators

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("payload", [False, True])
def test_stage_times_of_a_streamed_run(payload):
    """The stages' times add up to the call's, the time in the sink is the build's, and the last
    partition's and the levels above them are not left out."""
    tris = generators.icosphere(subdivisions=4, seed=6, payload=payload)
    with SvoContext(0) as ctx:
        for _ in range(2):  # (the second without allocations)
            calls = []
            t = time.perf_counter()
            info = ctx.run_stream(tris, payload, 256, lambda kind, b: (calls.append(kind), time.sleep(0.01)),
                                  memory_limit_mb=2)
            wall = (time.perf_counter() - t) * 1e3
        assert info.n_partitions == 8 and len(calls) >= 10
        sink = 10.0 * (len(calls) - 1)  # (the leading records go out before the first pass)
        assert sink - 0.5 <= info.ms_build <= wall
        assert info.ms_partition > 0 and info.ms_voxelize > 0
        assert info.ms_partition + info.ms_voxelize + info.ms_build <= wall
