"""Cases that measure the library: meshes in, octrees out, through its public calls.

Forms of a case:
  * "run":   one mesh resident in a context, the whole pipeline (partition, voxelize every
             partition, build) as svo_run does it, the records copied to device arrays;
  * "batch": many meshes in one svo_batch_run, used in place from device memory;
  * "host":  a mesh in host memory in, the octree's records in host memory out.

Meshes are made on the GPU from the seed: a noisy icosphere (20 * 4**size triangles, each
shared vertex displaced radially), an fBm heightfield of size x size vertices, or a soup of
'size' triangles on the surfaces of spheres; the shapes of ooc_svo_builder_amd.generators.
Outputs are the octree's records as they would be written to .octreenodes (three 64-bit
words a node) and .octreedata (eight 32-bit words a record), copied into the program's own
arrays (their size does not depend on the seed; the rest stays zero): bytes of a file format,
equal bit for bit or wrong.
"""
import functools
import math

import numpy as np
import torch

from ooc_svo_builder_amd import SvoContext, generators

BBOX = (0.0, 0.0, 0.0, 1.0, 1.0, 1.0)
MODEL, FIXED, LINEAR, NORMAL = 0, 1, 2, 3


def _case(name, form="run", mesh="terrain", size=0, payload=False, grid=256, limit_mb=2048,
          color=MODEL, levels=False, jobs=0, mix=0, max_tris=0):
    c = {"form": form, "mesh": mesh, "size": size, "payload": payload, "grid": grid,
         "limit_mb": limit_mb, "color": color, "levels": levels}
    if form == "batch":
        c = {"form": form, "jobs": jobs, "mix": mix, "max_tris": max_tris}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest useful call (a preview, a unit of a tool's pipeline): launches and
        # host waits are all of it
        _case("icosphere3_g64", mesh="icosphere", size=3, grid=64),
        # a small model at a preview resolution
        _case("icosphere5_g256", mesh="icosphere", size=5, grid=256),
        # a mid-size coloured scan with an odd vertex count, colours from normals
        _case("terrain401_g512_normal", size=401, payload=True, grid=512, color=NORMAL),
        # a large coloured scan with model colours, about a triangle per voxel
        _case("terrain1025_g1024_payload", size=1025, payload=True, grid=1024),
        # the geometry-only headline: 2,097,152 triangles at 2048 in one partition
        _case("terrain1025_g2048", size=1025, grid=2048, limit_mb=8192),
        # a low-polygon model at a high resolution: few triangles of thousands of columns
        _case("icosphere5_g2048", mesh="icosphere", size=5, grid=2048, limit_mb=8192),
        # a rough coloured surface: steep triangles of tens of columns, every voxel with a
        # record
        _case("icosphere7_g1024_payload", mesh="icosphere", size=7, payload=True, grid=1024),
        # out of core: 8 partitions (lists per partition, the streamed build), triangles of
        # log-normal sizes
        _case("soup6m_g4096_8parts", mesh="soup", size=6000000, grid=4096, limit_mb=8192),
        # -levels: averaged records for every internal node, for level-of-detail viewers
        _case("terrain701_g512_levels", size=701, payload=True, grid=512, levels=True),
        # asset conversion: many meshes of mixed kinds, sizes and grids at once
        _case("batch64_mix", form="batch", jobs=64, mix=4, max_tris=2000000),
        # host memory in, host memory out: a program without GPU buffers of its own
        _case("host_terrain300_g256", form="host", size=300, payload=True, grid=256),
    ]


def draw(rng):
    """Another case of the same ranges: 1e3 to 2.1e6 triangles (a soup: to 6e6), grids 64 to
    2048 (split into 8 partitions now and then), payload, colour modes and -levels."""
    kind = rng.random()
    if kind < 0.15:
        return _case("", form="batch", jobs=rng.randint(5, 64), mix=rng.randint(5, 1 << 20),
                     max_tris=int(math.exp(rng.uniform(math.log(5e4), math.log(1e6)))))
    grid = 1 << rng.randint(6, 11)
    payload = rng.random() < 0.4
    color = rng.choice((MODEL, MODEL, FIXED, LINEAR, NORMAL)) if payload else MODEL
    tris = math.exp(rng.uniform(math.log(1e3), math.log(2.1e6)))
    if kind < 0.25:
        return _case("", form="host", size=int(math.sqrt(min(tris, 3e5) / 2.0)) + 2,
                     payload=payload, grid=min(grid, 512), color=color)
    # one partition, or (a quarter of the draws) a limit that splits the grid into 8
    mb = max(2, grid ** 3 >> 20)
    limit = max(2, mb // 8) if rng.random() < 0.25 else max(2048, mb)
    levels = rng.random() < 0.15
    if levels or payload:
        grid = min(grid, 1024)
    mesh = rng.choice(("terrain", "terrain", "icosphere", "soup"))
    if mesh == "terrain":
        size = int(math.sqrt(tris / 2.0)) + 2
    elif mesh == "icosphere":
        size = min(7, max(3, round(math.log(tris / 20.0, 4))))
        if size >= 6:
            grid = min(grid, 1024)
    else:
        size = int(min(6e6, 3 * tris))
    return _case("", mesh=mesh, size=size, payload=payload and mesh != "soup", grid=grid,
                 limit_mb=limit, color=color if mesh != "soup" else MODEL, levels=levels)


# ---------------------------------------------------------------- meshes
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _uniform(g, shape, lo=0.0, hi=1.0):
    return torch.rand(shape, generator=g, device="cuda", dtype=torch.float64) * (hi - lo) + lo


def _records(p, tri, normals, colors):
    """(N, 9) records of vertices p and triangles tri, or (N, 21) with the normalized mean
    of the vertex normals and the vertex colours."""
    geo = p.float()[tri].reshape(len(tri), 9)
    if normals is None:
        return geo.contiguous()
    m = normals[tri].mean(dim=1)
    m = (m / m.norm(dim=1, keepdim=True)).float()
    return torch.cat([geo, m, colors.float()[tri].reshape(len(tri), 9)], dim=1).contiguous()


def _terrain(n, seed, payload):
    """z = 0.2 + 0.3 * fBm (six octaves of value noise from 4 cells on) over [0, 1]^2."""
    g = _generator(seed)
    ax = torch.linspace(0.0, 1.0, n, device="cuda", dtype=torch.float64)
    z = torch.zeros((n, n), device="cuda", dtype=torch.float64)
    for o in range(6):
        cells = 4 << o
        v = _uniform(g, (cells + 2, cells + 2))
        i = (ax * cells).floor().long()
        f = ax * cells - i
        s = f * f * (3.0 - 2.0 * f)
        rows = v[i] + (v[i + 1] - v[i]) * s[:, None]
        z += 0.5 ** o * (rows[:, i] + (rows[:, i + 1] - rows[:, i]) * s[None, :])
    z = 0.2 + 0.3 * z / sum(0.5 ** o for o in range(6))
    x, y = torch.meshgrid(ax, ax, indexing="ij")
    p = torch.stack([x, y, z], dim=-1).reshape(-1, 3)
    a = (torch.arange(n - 1, device="cuda")[:, None] * n + torch.arange(n - 1, device="cuda")).reshape(-1)
    # two triangles a cell, next to each other
    tri = torch.stack([a, a + n, a + n + 1, a, a + n + 1, a + 1], dim=1).reshape(-1, 3)
    if not payload:
        return _records(p, tri, None, None)
    dzdx, dzdy = torch.gradient(z, spacing=1.0 / (n - 1))
    nrm = torch.stack([-dzdx, -dzdy, torch.ones_like(z)], dim=-1).reshape(-1, 3)
    return _records(p, tri, nrm / nrm.norm(dim=1, keepdim=True), _uniform(g, (n * n, 3)))


@functools.lru_cache(maxsize=None)
def _sphere(subdivisions):
    """Unit icosphere: vertices and triangles (the same for every seed)."""
    t = (1.0 + 5.0 ** 0.5) / 2.0
    v = torch.tensor([[-1, t, 0], [1, t, 0], [-1, -t, 0], [1, -t, 0], [0, -1, t], [0, 1, t],
                      [0, -1, -t], [0, 1, -t], [t, 0, -1], [t, 0, 1], [-t, 0, -1], [-t, 0, 1]],
                     dtype=torch.float64, device="cuda")
    v = v / v.norm(dim=1, keepdim=True)
    f = torch.tensor([[0, 11, 5], [0, 5, 1], [0, 1, 7], [0, 7, 10], [0, 10, 11], [1, 5, 9],
                      [5, 11, 4], [11, 10, 2], [10, 7, 6], [7, 1, 8], [3, 9, 4], [3, 4, 2],
                      [3, 2, 6], [3, 6, 8], [3, 8, 9], [4, 9, 5], [2, 4, 11], [6, 2, 10],
                      [8, 6, 7], [9, 8, 1]], device="cuda")
    for _ in range(subdivisions):
        e = torch.cat([f[:, [0, 1]], f[:, [1, 2]], f[:, [2, 0]]]).sort(dim=1).values
        key, inv = torch.unique(e[:, 0] * (1 << 32) + e[:, 1], return_inverse=True)
        mid = v[key >> 32] + v[key & 0xFFFFFFFF]
        a, b, c = (len(v) + inv).reshape(3, -1)
        f = torch.cat([torch.stack(q, 1) for q in ((f[:, 0], a, c), (f[:, 1], b, a),
                                                   (f[:, 2], c, b), (a, b, c))])
        v = torch.cat([v, mid / mid.norm(dim=1, keepdim=True)])
    return v, f


def _icosphere(subdivisions, seed, payload):
    """Radius 0.4 around the grid's centre, vertices displaced radially by up to 0.02."""
    g = _generator(seed)
    v, f = _sphere(subdivisions)
    p = v * (0.4 + _uniform(g, (len(v), 1), -0.02, 0.02)) + 0.5
    return _records(p, f, v if payload else None, _uniform(g, (len(v), 3)) if payload else None)


def _soup(n, seed):
    """Equilateral triangles tangent to 200 spheres picked by area, edge lengths log-normal
    with a median of 4/8192."""
    g = _generator(seed)
    centers = _uniform(g, (200, 3), 0.1, 0.9)
    radii = _uniform(g, (200,), math.log(0.01), math.log(0.2)).exp()
    cdf = torch.cumsum(radii ** 2, 0)
    sid = torch.searchsorted(cdf, _uniform(g, (n,)) * cdf[-1]).clamp_(max=199)

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    d = normal(n, 3)
    d = d / d.norm(dim=1, keepdim=True)
    ctr = centers.float()[sid] + d * radii.float()[sid, None]
    pole = torch.where(d[:, :1].abs() < 0.9, torch.tensor([[1.0, 0.0, 0.0]], device="cuda"),
                       torch.tensor([[0.0, 1.0, 0.0]], device="cuda"))
    t1 = torch.linalg.cross(d, pole)
    t1 = t1 / t1.norm(dim=1, keepdim=True)
    t2 = torch.linalg.cross(d, t1)
    rad = 4.0 / 8192.0 / math.sqrt(3.0) * normal(n).exp()
    theta = _uniform(g, (n,)).float() * (2.0 * math.pi)
    out = torch.empty((n, 9), dtype=torch.float32, device="cuda")
    for k in range(3):
        ang = theta + 2.0 * math.pi * k / 3.0
        out[:, 3 * k:3 * k + 3] = ctr + (rad * ang.cos())[:, None] * t1 + (rad * ang.sin())[:, None] * t2
    return out


def _mesh(mesh, size, payload, seed):
    if mesh == "terrain":
        return _terrain(size, seed, payload)
    if mesh == "icosphere":
        return _icosphere(size, seed, payload)
    return _soup(size, seed)


def _mix(case):
    """The batch's meshes: kinds, sizes, payload and grids of generators.mix_spec."""
    return generators.mix_spec(case["jobs"], seed=case["mix"], n_max=case["max_tris"])


# ---------------------------------------------------------------- the calls
def prepare(case, seed):
    """The mesh (or meshes), a context, and the program's own arrays for the records."""
    torch.cuda.init()
    state = {"case": dict(case)}
    if case["form"] == "batch":
        state["jobs"] = [dict(records=_mesh(kind, size, payload, seed * 1000 + k),
                              payload=payload, gridsize=grid)
                         for k, (kind, size, payload, grid, _) in enumerate(_mix(case))]
    else:
        records = _mesh(case["mesh"], case["size"], case["payload"], seed)
        if case["form"] == "host":
            state["records"] = records.cpu().numpy()
    n_nodes, n_data = _room(case)
    if case["form"] == "host":
        state["nodes"] = np.zeros((n_nodes, 3), np.int64)
        state["data"] = np.zeros((n_data, 8), np.int32)
    else:
        state["nodes"] = torch.zeros((n_nodes, 3), dtype=torch.int64, device="cuda")
        state["data"] = torch.zeros((n_data, 8), dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    ctx = state["ctx"] = SvoContext(0)
    if case["form"] == "run":
        ctx.load_mesh(records, case["payload"])
    return state


def run(state):
    case, ctx, nodes, data = state["case"], state["ctx"], state["nodes"], state["data"]
    if case["form"] == "batch":
        results, info = ctx.batch_run(state["jobs"])
        counts = np.array([(r.n_nodes, r.n_data, r.node_offset, r.data_offset, r.nfilled,
                            r.n_partitions, r.hazard) for r in results], dtype=np.int64)
    else:
        options = dict(memory_limit_mb=case["limit_mb"], bbox=BBOX, color_mode=case["color"],
                       levels=case["levels"])
        if case["form"] == "host":
            info = ctx.run(state["records"], case["payload"], case["grid"], **options)
        else:
            info = ctx.rerun(case["payload"], case["grid"], **options)
        counts = np.array([info.n_nodes, info.n_data, info.nfilled, info.hazard], dtype=np.int64)
    if info.n_nodes > len(nodes) or info.n_data > len(data):
        raise RuntimeError("the octree is larger than the arrays for it")
    host = case["form"] == "host"
    ctx.copy_nodes_to(nodes.ctypes.data if host else nodes.data_ptr(), 0, info.n_nodes)
    ctx.copy_data_to(data.ctypes.data if host else data.data_ptr(), 0, info.n_data)
    return counts, nodes, data


def exact(case, seed):
    """Every output is a count or a record's bytes: none has a value in 64-bit arithmetic.
    Which voxels a triangle covers, and the bits of a voxel's colour, are defined by the
    file format's FP32 evaluation order."""
    return None


# ---------------------------------------------------------------- the work of a pass
def _triangles(mesh, size):
    return {"terrain": 2 * (size - 1) ** 2, "icosphere": 20 * 4 ** size, "soup": size}[mesh]


def _voxels(mesh, size, grid):
    """Occupied voxels, from counts of these generators over their ranges."""
    if mesh == "terrain":
        return 1.9 * grid ** 2
    if mesh == "icosphere":  # the spikes' area, within the 0.04 thick shell they fill
        area = 3.0 * math.sqrt(1.0 + (0.046 * 2 ** size) ** 2)
        return min(area, 0.08 * grid + 3.0) * grid ** 2
    # a soup: its triangles' voxels while they are sparse, at most its spheres' surfaces
    edge = grid * 4.0 / 8192.0  # the median, in voxels
    each = 1.0 + 3.2 * edge + 4.7 * edge ** 2
    sheets = 22.0 * grid ** 2
    return sheets * (1.0 - math.exp(-size * each / sheets))


def _parts(case):
    if case["form"] == "batch":
        return [(kind, size, payload, grid, False) for kind, size, payload, grid, _ in _mix(case)]
    return [(case["mesh"], case["size"], case["payload"], case["grid"], case["levels"])]


def _counts(case):
    """(nodes, data records): an octree of a surface has about a third more nodes than
    voxels (a soup's up to 2.7 times as many where its triangles are far apart); a record per
    voxel with payload, and per inner node with -levels."""
    nodes = data = 0.0
    for mesh, size, payload, grid, levels in _parts(case):
        v = _voxels(mesh, size, grid)
        inner = v / 3
        if mesh == "soup":
            inner += 1.35 * v * math.exp(-v / (3.5 * grid ** 2))
        nodes += v + inner
        data += (v if payload else 2) + (inner if levels else 0)
    return nodes, data


def _room(case):
    """Room for the records whatever the seed: geometry-only meshes have two data records,
    everything else up to its estimate and more than half."""
    nodes, data = _counts(case)
    exact_data = not any(payload or levels for _, _, payload, _, levels in _parts(case))
    return int(1.6 * nodes) + 65536, int(data) if exact_data else int(1.6 * data) + 65536


def work(case):
    """Each triangle record read once, each node and data record written once."""
    nodes, data = _counts(case)
    mesh_bytes = sum(_triangles(mesh, size) * (84 if payload else 36)
                     for mesh, size, payload, _, _ in _parts(case))
    return {"bytes": mesh_bytes + 24 * nodes + 32 * data, "flops": 0.0}
