"""The voxelizer's linear classification of column runs against the tests it stands for.

svo_walk.h answers "every voxel of this run passes" or "none outside it does" from bounds
with an error term, and leaves the rest to the reference's FP32 tests
(voxelizer.cpp:257-287). Compiled for the host, it is compared here voxel by voxel with
those tests: no certain answer may differ, whatever the triangle's orientation, alignment,
scale or clamp box."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("walk") / "walk_check.so")
    subprocess.run([HIPCC, "--offload-host-only", "-O2", "-std=c++17", "-fPIC", "-shared",
                    "-ffp-contract=off", "-fno-fast-math",
                    os.path.join(ROOT, "tests", "native", "walk_check.hip"), "-o", so], check=True)
    lib = C.CDLL(so)

    def run(tris, G, unit=None, pmin=(0, 0, 0), pmax=None):
        tris = np.ascontiguousarray(tris, np.float32)
        out = (C.c_uint64 * 6)()
        lib.walk_check(tris.ctypes.data_as(C.c_void_p), C.c_uint64(len(tris)),
                       C.c_float(np.float32(1.0 / G if unit is None else unit)), C.c_uint64(G),
                       (C.c_int * 3)(*pmin), (C.c_int * 3)(*(pmax or (G - 1,) * 3)), out)
        return dict(zip(("voxels", "wrong", "columns", "uncertain", "careful", "accepted"), out))
    return run


def _random(rng, n, size, lo=0.0, hi=1.0):
    c = rng.uniform(lo, hi, (n, 1, 3))
    return (c + rng.normal(size=(n, 3, 3)) * size).reshape(n, 9).astype(np.float32)


@pytest.mark.parametrize("G", [64, 1024, 2048, 32768])
@pytest.mark.parametrize("kind", ["small", "large", "top corner", "odd unit", "clamped"])
def test_certain_answers_are_the_tests_answers(check, G, kind):
    rng = np.random.default_rng([G, len(kind)])
    kw = {}
    tris = _random(rng, 8000, 3.0 / G)
    if kind == "large":
        tris = _random(rng, 600, 12.0 / G)
    elif kind == "top corner":  # the largest coordinates
        tris = _random(rng, 8000, 3.0 / G, 0.98, 1.0)
    elif kind == "odd unit":  # not a power of two; part of the triangles outside the grid
        kw["unit"] = 0.77777779 / G
    elif kind == "clamped":  # a partition's box
        kw.update(pmin=(G // 2, 0, 0), pmax=(G - 1, G // 2 - 1, G // 2 - 1))
    got = check(tris, G, **kw)
    assert got["wrong"] == 0, got
    assert got["accepted"] > 0
    if G <= 2048:  # the classification does the work: few columns are left to the tests
        assert got["uncertain"] < 0.05 * got["columns"], got


@pytest.mark.parametrize("G", [64, 2048])
@pytest.mark.parametrize("kind", ["voxel corners", "flat", "edge along an axis", "two equal vertices",
                                  "collinear", "sliver", "tiny scale", "huge scale", "overflow",
                                  "nan and infinity", "negative unit"])
def test_degenerate_and_aligned_triangles(check, G, kind):
    rng = np.random.default_rng([G, len(kind), 7])
    t = _random(rng, 3000, 4.0 / G)
    unit = 1.0 / G
    if kind == "voxel corners":  # bounds on integers throughout
        t = (np.round(t * G) / G).astype(np.float32)
    elif kind == "flat":
        t = (np.round(t * G) / G).astype(np.float32)
        t[:, 2] = t[:, 5] = t[:, 8]
    elif kind == "edge along an axis":
        t[:, 0] = t[:, 3]
    elif kind == "two equal vertices":
        t[:, 3:6] = t[:, 0:3]
    elif kind == "collinear":
        t[:, 6:9] = t[:, 0:3] + (t[:, 3:6] - t[:, 0:3]) * np.float32(0.5)
    elif kind == "sliver":
        t = (_random(rng, 1000, 1.0) * np.array([1e-3, 1e-6, 8.0 / G] * 3, np.float32)
             + np.float32(0.3)).astype(np.float32)
    elif kind == "tiny scale":
        t, unit = t * np.float32(1e-20), 1e-20 / G
    elif kind == "huge scale":
        t, unit = t * np.float32(1e20), 1e20 / G
    elif kind == "overflow":
        t, unit = t[:300] * np.float32(1e37), 1e37 / G
    elif kind == "nan and infinity":
        t = _random(rng, 60, 0.5 / G) if G > 64 else t[:300]
        t[::3, 4] = np.nan
        t[1::3, 7] = np.inf
        if G > 64:  # (bboxes reach the grid's top: a small box of it)
            got = check(t, G, pmin=(0, 0, 0), pmax=(63, 63, 63))
            assert got["wrong"] == 0, got
            return
    elif kind == "negative unit":
        unit = -1.0 / G
    got = check(t, G, unit=unit)
    assert got["wrong"] == 0, got
