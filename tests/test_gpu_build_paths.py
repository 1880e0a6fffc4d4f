"""Branches of the build, the payload marks, the partition lists and the record copies at the
sizes where they change, against the oracle (bit for bit: every output is a count or bytes of
a file format)."""
import numpy as np
import pytest

import oracle
from ooc_svo_builder_amd import SvoContext, generators

pytestmark = pytest.mark.gpu


def _mesh(rng, n, size, payload=False, spread=0.4):
    c = 0.5 + rng.uniform(-spread, spread, (n, 1, 3))
    geo = (c + rng.normal(size=(n, 3, 3)) * size).reshape(n, 9).astype(np.float32)
    return np.concatenate([geo, rng.uniform(0, 1, (n, 12)).astype(np.float32)], 1) if payload else geo


def _same(ctx, info, tris, payload, G, limit=2048):
    nodes, data, hz, parts, nf = oracle.pipeline(tris, payload, G, limit)
    assert (info.n_nodes, info.n_data, info.nfilled, info.hazard, info.n_partitions) == \
        (len(nodes), len(data), nf, hz, parts)
    assert ctx.nodes(info.n_nodes).tobytes() == nodes.tobytes()
    assert ctx.data(info.n_data).tobytes() == data.tobytes()


@pytest.mark.parametrize("payload", [False, True])
@pytest.mark.parametrize("G,n", [(16, 3), (32, 1), (128, 250), (256, 1023), (256, 1024), (256, 1025),
                                 (1024, 1500), (1024, 700), (1024, 4096), (1024, 4097)])
def test_bricks_around_the_upper_levels_paths(G, n, payload):
    """A triangle in each of n bricks (all of 16^3): the upper levels in one block with the nodes in LDS (up to 1024 bricks, 2816 nodes) or
    by launches, the records staged (past 4096 bricks) or not."""
    rng = np.random.default_rng(n)
    side = G // 16
    at = rng.choice(side ** 3, min(n, side ** 3), replace=False)
    xyz = np.stack([at % side, at // side % side, at // side // side], 1) * 16 + \
        rng.integers(1, 15, (len(at), 3))
    p = (xyz[:, None, :] + 0.5) / G + np.array([[0, 0, 0], [0.2, 0, 0], [0, 0.2, 0]]) / G
    tris = p.reshape(-1, 9).astype(np.float32)
    if payload:
        tris = np.concatenate([tris, rng.uniform(0, 1, (len(tris), 12)).astype(np.float32)], 1)
    with SvoContext(0) as ctx:
        _same(ctx, ctx.run(tris, payload, G), tris, payload, G)


def test_small_jobs_of_a_batch():
    """Few bricks over several jobs: empty ones, ones of a single brick, of different depths."""
    rng = np.random.default_rng(1)
    jobs = []
    for G, n, payload in ((16, 4, False), (64, 30, True), (32, 0, False), (256, 60, False),
                          (16, 2, True), (128, 25, True), (64, 0, True)):
        jobs.append(dict(records=_mesh(rng, n, 2.0 / G, payload), payload=payload, gridsize=G))
    with SvoContext(0) as ctx:
        for _ in range(3):  # the second is replayed from graphs
            res, info = ctx.batch_run(jobs)
            nodes, data = ctx.nodes(info.n_nodes), ctx.data(info.n_data)
            for q, r in zip(jobs, res):
                w_nodes, w_data, hz, _, nf = oracle.pipeline(q["records"], q["payload"], q["gridsize"], 2048)
                assert (r.n_nodes, r.n_data, r.nfilled, r.hazard) == (len(w_nodes), len(w_data), nf, hz)
                assert nodes[r.node_offset:r.node_offset + r.n_nodes].tobytes() == w_nodes.tobytes()
                assert data[r.data_offset:r.data_offset + r.n_data].tobytes() == w_data.tobytes()


@pytest.mark.parametrize("graphs", [False, True])
@pytest.mark.parametrize("payload", [False, True])
@pytest.mark.parametrize("G,n", [(16, 3), (64, 30), (256, 60), (512, 4000)])
def test_a_batch_of_one_job(G, n, payload, graphs):
    """Its descriptor is the uploaded one, with graphs or without, on few bricks and on many."""
    tris = _mesh(np.random.default_rng(n), n, 2.0 / G, payload)
    w_nodes, w_data, hz, _, nf = oracle.pipeline(tris, payload, G, 2048)
    with SvoContext(0) as ctx:
        ctx.set_graphs(graphs)
        for _ in range(3):
            (r,), info = ctx.batch_run([dict(records=tris, payload=payload, gridsize=G)])
            assert (r.n_nodes, r.n_data, r.nfilled, r.hazard) == (len(w_nodes), len(w_data), nf, hz)
            assert ctx.nodes(info.n_nodes).tobytes() == w_nodes.tobytes()
            assert ctx.data(info.n_data).tobytes() == w_data.tobytes()


@pytest.mark.parametrize("direct", [0, 16])
@pytest.mark.parametrize("order", ["as made", "shuffled", "doubled"])
@pytest.mark.parametrize("mesh", ["terrain", "spikes", "heap"])
def test_payload_winners(mesh, order, direct):
    """Lines of cells gathered in LDS: neighbouring triangles that share lines, steep ones of many
    lines each (more than a wave holds), and many triangles on the same few lines; the lowest
    triangle wins whatever the order."""
    G = 256
    rng = np.random.default_rng(7)
    if mesh == "terrain":
        tris = generators.terrain(n=150, seed=3, payload=True)
    elif mesh == "spikes":
        tris = _mesh(rng, 900, 12.0 / G, True)
    else:
        tris = _mesh(rng, 3000, 3.0 / G, True, spread=0.02)
    if order == "shuffled":
        tris = tris[rng.permutation(len(tris))]
    elif order == "doubled":
        tris = np.concatenate([tris[len(tris) // 2:], tris])
        tris[:, 9:] = rng.uniform(0, 1, (len(tris), 12)).astype(np.float32)
    tris = np.ascontiguousarray(tris)
    with SvoContext(0) as ctx:
        k = ctx.get_tuning()
        ctx.set_knobs(k[0], direct, k[2], k[3])
        _same(ctx, ctx.run(tris, True, G, 2048), tris, True, G)


def test_tiles_of_both_kinds_in_one_pass():
    """Geometry-only and payload units mixed by runs of tiles: one kind in a minority, runs that
    are not full, and payload units alone."""
    rng = np.random.default_rng(2)
    for counts in ([(5, False)] * 3 + [(7000, True)], [(9000, False)] + [(3, True)] * 2,
                   [(70, True), (900, True)], [(1100, False), (1025, True), (64, False), (65, True)]):
        jobs = [dict(records=_mesh(rng, n, 2.0 / 128, p), payload=p, gridsize=128) for n, p in counts]
        with SvoContext(0) as ctx:
            res, info = ctx.batch_run(jobs)
            nodes, data = ctx.nodes(info.n_nodes), ctx.data(info.n_data)
            for q, r in zip(jobs, res):
                w_nodes, w_data, _, _, nf = oracle.pipeline(q["records"], q["payload"], 128, 2048)
                assert (r.n_nodes, r.n_data, r.nfilled) == (len(w_nodes), len(w_data), nf)
                assert nodes[r.node_offset:r.node_offset + r.n_nodes].tobytes() == w_nodes.tobytes()
                assert data[r.data_offset:r.data_offset + r.n_data].tobytes() == w_data.tobytes()


@pytest.mark.parametrize("payload", [False, True])
def test_units_past_32_bits(payload):
    """A unit of 2^33 voxels takes 64-bit places, one of 2^30 (the same in 8 partitions) 32-bit
    ones; triangles in every octant, some of many columns."""
    G = 2048
    rng = np.random.default_rng(9)
    tris = np.concatenate([_mesh(rng, 150, 2.0 / G, payload, spread=0.49),
                           _mesh(rng, 20, 30.0 / G, payload)])
    want = oracle.pipeline(tris, payload, G, 1024)[:2]
    with SvoContext(0) as ctx:
        for limit in (8192, 1024):
            info = ctx.run(tris, payload, G, limit)
            assert ctx.nodes(info.n_nodes).tobytes() == want[0].tobytes()
            assert ctx.data(info.n_data).tobytes() == want[1].tobytes()


@pytest.mark.parametrize("payload", [False, True])
def test_a_mesh_that_covers_nothing(payload):
    """No brick is flagged: the scan that reads back has no element, and must still do it; the
    next mesh of the same context is not affected."""
    G = 64
    rng = np.random.default_rng(4)
    none, some = _mesh(rng, 100, 2.0 / G, payload), _mesh(rng, 100, 2.0 / G, payload)
    none[:, 3] = 1e12  # a bbox that ends before it starts
    with SvoContext(0) as ctx:
        for tris in (none, some, none):
            _same(ctx, ctx.run(tris, payload, G), tris, payload, G)


@pytest.mark.parametrize("n_parts", [8, 64, 512])
@pytest.mark.parametrize("n", [1, 64, 2047, 2048, 2049, 300001])
def test_partition_lists(n_parts, n):
    """All lists at once (up to 64 partitions) around a tile's 2048 triangles, with triangles
    that touch every partition, none, and NaN; 512 partitions go one by one."""
    G = 128
    rng = np.random.default_rng(n)
    tris = _mesh(rng, n, 0.02, spread=0.5)
    tris[::50] = rng.uniform(-1, 2, (len(tris[::50]), 9)).astype(np.float32)
    tris[7::100] += 5.0
    tris[11::500, 4] = np.nan
    _, want = oracle.partition(tris, False, (0, 0, 0, 1, 1, 1), G, n_parts)
    with SvoContext(0) as ctx:
        ctx.load_mesh(tris, False)
        counts = ctx.partition(1.0 / G, G, n_parts)
        assert [len(w) for w in want] == list(counts)
        for j, w in enumerate(want):
            assert np.array_equal(ctx.partition_indices(j, int(counts[j])), w)


def test_copies_of_record_ranges():
    """Copies to device memory around the size up to which a copy raises its own flag (2 MB),
    of even and odd counts, one after the other; and the same ranges to host memory."""
    import torch
    tris = generators.icosphere(subdivisions=5, seed=2, payload=True)
    with SvoContext(0) as ctx:
        info = ctx.run(tris, True, 256)
        nodes = ctx.nodes(info.n_nodes)
        want = torch.from_numpy(nodes.view(np.int64).reshape(-1, 3).copy())
        assert info.n_nodes > 200000
        for count in (1, 2, 3, 1000, 21845, 21846, 43690, 43691, 87380, 87381, 87382, 87383, 200000):
            for first in (0, 1, 777):
                dst = torch.full((count + 2, 3), -1, dtype=torch.int64, device="cuda")
                torch.cuda.synchronize()
                ctx.copy_nodes_to(dst[1:].data_ptr(), first, count)
                got = dst.cpu()
                assert torch.equal(got[1:count + 1], want[first:first + count])
                assert (got[0] == -1).all() and (got[-1] == -1).all()
                host = np.full((count + 2, 3), -1, np.int64)
                ctx.copy_nodes_to(host[1:].ctypes.data, first, count)
                assert np.array_equal(host[1:-1], want[first:first + count].numpy())
                assert (host[0] == -1).all() and (host[-1] == -1).all()
