"""What the voxelizer keeps on the device between passes, when an allocation fails.

Its brick table, word flags, cells and slots are zero whenever no pass is running, and the
context remembers how much of each is. A pass that grows them and then fails, or that fails
with marks in them, must leave that knowledge right for the next one: the server runs the jobs
of a failed batch one by one on the same context. The library's host side is compiled here
against a stand-in for the device (tests/native/device_state_check.hip), where every
allocation of a pass fails in turn and the passes that follow are checked."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from ooc_svo_builder_amd import lib as binding

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "ooc_svo_builder_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
NAMES = ("allocations", "unclean", "outside", "bad_grid", "marks", "dense", "stale")


@pytest.fixture(scope="module")
def device(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("state")
    src = [os.path.join(ROOT, "tests", "native", "device_state_check.hip")] + \
        [os.path.join(CSRC, f) for f in ("svo_build.hip", "svo_stream.hip", "svo_capi.hip")]
    runs, objs = [], []
    for f in src:
        objs.append(str(tmp / (os.path.basename(f) + ".o")))
        runs.append(subprocess.Popen([HIPCC, "--offload-host-only", "-O1", "-std=c++17", "-fPIC",
                                      "-ffp-contract=off", "-fno-fast-math", "-c", f, "-o", objs[-1]]))
    assert [r.wait() for r in runs] == [0] * len(runs)
    so = str(tmp / "device_state.so")
    # (no code for a device is linked in: the registration's references to it are null)
    names = subprocess.run(["nm", "-u"] + objs, check=True, capture_output=True, text=True).stdout
    none = ["-Wl,--defsym=%s=0" % w for w in set(names.split()) if w.startswith("__hip_fatbin")]
    subprocess.run(["g++", "-shared", "-o", so] + objs + ["-Wl,-Bsymbolic", "-lpthread"] + none, check=True)
    L = C.CDLL(so)
    for name, (res, args) in binding.SIGNATURES.items():
        if hasattr(L, name):
            getattr(L, name).restype, getattr(L, name).argtypes = res, args
    return L


def _arm(L, fail_at=-1, n_occ=5, n_vox=100):
    L.state_arm(C.c_long(fail_at), C.c_uint64(n_occ), C.c_uint64(n_vox))


def _state(L):
    out = (C.c_uint64 * 7)()
    L.state_read(out)
    return dict(zip(NAMES, out))


def _mesh(payload, n=40):
    return np.zeros((n, 21 if payload else 9), np.float32)


def _pass(L, ctx, payload, G):
    t = _mesh(payload)
    rc = L.svo_mesh_load(ctx, t.ctypes.data_as(C.c_void_p), len(t), int(payload), 0)
    return rc or L.svo_voxelize(ctx, 0, 0, G ** 3, 1.0 / G, G, 0, None)


def _batch(L, ctx, G, kinds):
    jobs, res, info = (binding.Job * len(kinds))(), (binding.JobResult * len(kinds))(), binding.RunInfo()
    keep = [binding.fill_job(q, dict(records=_mesh(p), payload=p, gridsize=G))
            for q, p in zip(jobs, kinds)]
    rc = L.svo_batch_run(ctx, jobs, len(kinds), res, C.byref(info))
    del keep
    return rc


def _find(L, n_occ):
    L.state_found(C.c_uint64(n_occ), C.c_uint64(20 * n_occ))


def _fail_each(L, first, grown, after, marked, dense_mb=None):
    """Passes 'first' on a new context, then 'grown' with its k-th allocation failing, then the
    passes 'after', for every k up to the allocations it makes. marked: the failures after its
    marks, else those before them."""
    failed = 0
    for k in range(100):
        ctx = C.c_void_p()
        L.state_clear()
        _arm(L)
        assert L.svo_ctx_create(0, C.byref(ctx)) == 0
        assert L.svo_ctx_set_graphs(ctx, 0) == 0
        if dense_mb is not None:
            assert L.svo_ctx_set_tuning(ctx, 0, dense_mb) == 0
        for f in first:
            assert f(ctx) == 0, k
        _arm(L, fail_at=k)
        marks = _state(L)["marks"]
        rc = grown(ctx)
        s = _state(L)
        if s["allocations"] <= k:  # it made fewer
            assert rc == 0 and failed >= 1
            L.svo_ctx_destroy(ctx)
            return
        assert rc in (binding.SVO_ERR_NOMEM, binding.SVO_ERR_DEVICE), (k, rc)
        if marked == (s["marks"] > marks):
            failed += 1
            _arm(L)
            for f in after:
                assert f(ctx) == 0, k
            s = _state(L)
            assert (s["unclean"], s["outside"], s["bad_grid"], s["stale"]) == (0, 0, 0, 0), (k, s)
        L.svo_ctx_destroy(ctx)
    raise AssertionError("the pass still allocates after 100 allocations")


def _passes(L, kinds, dense, marked):
    a, b = kinds
    _fail_each(L, [lambda c: _pass(L, c, a, 32)], lambda c: (_find(L, 400), _pass(L, c, b, 128))[1],
               [lambda c: _pass(L, c, a, 32), lambda c: _pass(L, c, b, 32), lambda c: _pass(L, c, b, 64),
                lambda c: _pass(L, c, a, 64), lambda c: _pass(L, c, b, 128)],
               marked, None if dense else 0)


def _batches(L, marked):
    kinds = (False, True, False)
    _fail_each(L, [lambda c: _batch(L, c, 32, kinds)], lambda c: (_find(L, 400), _batch(L, c, 128, kinds))[1],
               [lambda c: _batch(L, c, 32, kinds), lambda c: _batch(L, c, 128, (False,)),
                lambda c: _batch(L, c, 128, (True,)), lambda c: _batch(L, c, 128, kinds)], marked)


KINDS = [(False, False), (True, True), (False, True), (True, False)]


@pytest.mark.parametrize("dense", [True, False])
@pytest.mark.parametrize("kinds", KINDS)
def test_a_pass_that_fails_as_it_grows(device, kinds, dense):
    """A pass, a larger one that fails before its marks, the first again, one in between and the
    larger again: nothing that was replaced is taken for zero."""
    _passes(device, kinds, dense, marked=False)


def test_a_batch_that_fails_as_it_grows(device):
    """The server's order: the batch fails, then its jobs run one by one on the same context."""
    _batches(device, marked=False)


@pytest.mark.parametrize("kinds,dense", [(k, d) for k in KINDS for d in (True, False) if k[1] or not d])
def test_a_pass_that_fails_with_marks(device, kinds, dense):
    """The same with failures after the marks (the records' array above all; a dense geometry-only
    pass allocates nothing then): what they left is cleared before the next marks."""
    _passes(device, kinds, dense, marked=True)


def test_a_batch_that_fails_with_marks(device):
    _batches(device, marked=True)


def test_slots_that_fail_to_grow(device):
    """A pass on touched bricks that needs more slots than there are (1500 of 1024)."""
    L = device
    _fail_each(L, [lambda c: _pass(L, c, False, 256)],
               lambda c: (_find(L, 1500), _pass(L, c, False, 256))[1],
               [lambda c: _pass(L, c, False, 64), lambda c: _pass(L, c, True, 256)], True, 0)


@pytest.mark.parametrize("gib", [1, 63, 64, 65, 128, 200])
def test_copies_of_any_size(device, gib):
    """A record copy's grid is one that HIP takes (less than 2^32 threads)."""
    L = device
    for bytes_ in ((gib << 30) - 24, gib << 30, (gib << 30) + 24):
        L.state_clear()
        assert L.state_copy(C.c_uint64(bytes_)) == 0
        assert _state(L)["bad_grid"] == 0


@pytest.mark.parametrize("n_vox", [1 << 31, (1 << 31) + 1, 0xFFFFFF00, 0xFFFFFF01, 0xFFFFFFF0])
def test_payload_records_of_almost_two_to_the_32_voxels(device, n_vox):
    """The records of a pass on touched bricks, up to the largest one that is accepted."""
    L, ctx = device, C.c_void_p()
    L.state_clear()
    _arm(L)
    assert L.svo_ctx_create(0, C.byref(ctx)) == 0
    assert L.svo_ctx_set_tuning(ctx, 0, 0) == 0
    L.state_found(C.c_uint64(500), C.c_uint64(n_vox))
    assert _pass(L, ctx, True, 256) == 0
    assert _state(L)["bad_grid"] == 0
    L.svo_ctx_destroy(ctx)


@pytest.mark.parametrize("G,payload", [(8192, False), (16384, False), (4096, True), (8192, True)])
def test_a_dense_limit_beyond_any_memory(device, G, payload):
    """A caller's limit does not make a pass dense whose bricks or cells have no 32-bit place."""
    L, ctx = device, C.c_void_p()
    L.state_clear()
    _arm(L)
    assert L.svo_ctx_create(0, C.byref(ctx)) == 0
    assert L.svo_ctx_set_tuning(ctx, 0, 1 << 40) == 0
    assert _pass(L, ctx, payload, G) == 0
    s = _state(L)
    assert (s["outside"], s["bad_grid"]) == (0, 0)
    assert s["dense"] == (G ** 3 <= 1 << (36 if payload else 39))
    L.svo_ctx_destroy(ctx)


@pytest.mark.parametrize("payload", [False, True])
def test_slots_that_grow(device, payload):
    """Passes on touched bricks that need more slots than there are: the redone pass goes through
    the new ones, and what it writes has room."""
    L, ctx = device, C.c_void_p()
    L.state_clear()
    _arm(L)
    assert L.svo_ctx_create(0, C.byref(ctx)) == 0
    assert L.svo_ctx_set_tuning(ctx, 0, 0) == 0
    for n_occ in (500, 1500, 40000, 90000, 2000):
        _find(L, n_occ)
        marks = _state(L)["marks"]
        assert _pass(L, ctx, payload, 1024) == 0
        s = _state(L)
        assert s["marks"] > marks and (s["unclean"], s["outside"], s["bad_grid"], s["stale"]) == (0, 0, 0, 0), (n_occ, s)
    L.svo_ctx_destroy(ctx)


def _run(L, ctx, payload, G, limit=2048, levels=0, n=40, sink=None):
    t, b, info = _mesh(payload, n), np.array([0, 0, 0, 1, 1, 1], np.float32), binding.RunInfo()
    p = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
    if sink is not None:
        return L.svo_run_stream(ctx, p(t), len(t), int(payload), 0, p(b), G, limit, 0, levels, sink, None,
                                C.byref(info))
    return L.svo_run(ctx, p(t), len(t), int(payload), 0, p(b), G, limit, 0, levels, C.byref(info))


@pytest.mark.parametrize("dense", [True, False])
def test_no_launch_is_given_memory_that_is_gone(device, dense):
    """Whole calls of growing and shrinking sizes on one context, each after every other."""
    L, ctx = device, C.c_void_p()
    L.state_clear()
    _arm(L)
    assert L.svo_ctx_create(0, C.byref(ctx)) == 0
    assert L.svo_ctx_set_graphs(ctx, 0) == 0
    if not dense:
        assert L.svo_ctx_set_tuning(ctx, 0, 0) == 0
    sink = binding.SINK_FN(lambda user, kind, p, n: 0)
    dst = np.zeros(1 << 20, np.uint8)
    codes = np.arange(5000, dtype=np.uint64)

    def added(c):
        t = _mesh(False, 0)
        rc = L.svo_mesh_load(c, t.ctypes.data_as(C.c_void_p), 0, 0, 0)
        rc = rc or L.svo_add_voxels(c, codes.ctypes.data_as(C.c_void_p), None, len(codes))
        return rc or L.svo_build(c, 64, 1, None, None, None)

    calls = [lambda c: _run(L, c, False, 64), lambda c: _run(L, c, True, 64), lambda c: _run(L, c, True, 128, levels=1),
             lambda c: _run(L, c, False, 128, 2, n=3000), lambda c: _run(L, c, True, 128, 2),
             lambda c: _run(L, c, True, 128, 2, 1), lambda c: _run(L, c, True, 128, 2, 0, 90, sink),
             lambda c: _batch(L, c, 64, (False, True)), lambda c: _batch(L, c, 128, (True, True, False)), added,
             lambda c: L.svo_copy_nodes(c, dst.ctypes.data_as(C.c_void_p), 0, 10)]
    step = 0
    for n_occ in (5, 1500, 90, 9000):
        for a in calls:
            for b in calls:
                _find(L, n_occ)
                for f in (a, b):
                    rc = f(ctx)
                    s = _state(L)
                    assert rc == 0 or f is calls[-1], (step, rc, L.svo_last_error())
                    assert (s["unclean"], s["outside"], s["bad_grid"], s["stale"]) == (0, 0, 0, 0), (step, s)
                    step += 1
        _find(L, 20 * n_occ)
    L.svo_ctx_destroy(ctx)
