"""Host code of the library against a stand-in HIP runtime (tests/hip_stub).

Each test runs in a process of its own (no GPU, no torch): the stand-in is
loaded first with RTLD_GLOBAL, so that libfdkhip.so's HIP calls come to it; it
logs launches and copies, keeps device memory on the host and lets chosen
calls fail.  Kernels do not run, so only what the host decides is tested:
devices, launch grids, layouts, error paths.
"""
from __future__ import annotations

import os
import subprocess
import sys
import textwrap

import pytest

from conftest import ROOT

STUB = os.path.join(ROOT, "tests", "hip_stub", "fake_hip.c")

PREAMBLE = """
import ctypes as C, sys, time
sys.path.insert(0, %(root)r)
fake = C.CDLL(%(stub)r, mode=C.RTLD_GLOBAL)
fake.fake_log.restype = C.c_char_p
fake.fake_fail.argtypes = [C.c_char_p, C.c_int]
fake.fake_fast_lds.argtypes = [C.c_size_t]
import numpy as np
from mirt_amd import _lib
lib = _lib.load()
F32, F16 = _lib.F32, _lib.F16

def log(kind=None):
    rows = [r.split() for r in fake.fake_log().decode().splitlines()]
    return [[int(x) for x in r[1:]] for r in rows if r[0] == kind] if kind else rows

def geom(nx, ny, nz, ns, nt, dx=1.0, dz=1.0, ds=1.0, dt=1.0):
    return _lib.Geom(nx, ny, nz, dx, -dx, dz, 0, 0, 0, 541.0, 949.0, float("inf"), ns, nt,
                     ds, dt, 0, 0)

def plan(g, na=24, fmt=F32):
    h, beta = C.c_void_p(), np.linspace(0, 6, na)
    _lib.check(lib.fdkhip_plan_create(C.byref(h), C.byref(g), na,
                                      C.c_void_p(beta.ctypes.data), None, fmt, 0))
    return h

BUF = C.c_void_p(1 << 20)   # a device buffer that no kernel reads
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("hip_stub") / "libfakehip.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-I/opt/rocm/include", "-o", out, STUB],
                   check=True)
    return out


def _run(stub, body):
    code = PREAMBLE % dict(root=ROOT, stub=stub) + textwrap.dedent(body) + "\nprint('passed')\n"
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.endswith("passed\n"), r.stdout + r.stderr


def test_count_updates_device_and_failures(stub):
    """The count of a plan whose shape needed no survey runs on the plan's own
    device and stream whichever device is current, goes back to that device,
    and stays unknown after a failure."""
    _run(stub, """
    fake.fake_fill(1)
    for fmt in (F32, F16):
        h, n = plan(geom(64, 64, 32, 128, 96), fmt=fmt), C.c_int64(-7)
        assert not log("launch")          # no survey
        fake.hipSetDevice(1)
        fake.fake_fail(b"hipStreamSynchronize", 1)
        assert lib.fdkhip_plan_count_updates(h, C.byref(n)) == -4 and n.value == -7
        fake.fake_clear()
        assert lib.fdkhip_plan_count_updates(h, C.byref(n)) == 0
        assert n.value == 0x0101010101010101
        rows = log("launch")
        assert rows and all(r[0] == 0 and r[-1] != 0 for r in rows), rows
        assert all(r[0] == 0 for r in log("memcpy"))
        d = C.c_int()
        fake.hipGetDevice(C.byref(d))
        assert d.value == 1
        fake.fake_clear()
        assert lib.fdkhip_plan_count_updates(h, C.byref(n)) == 0 and not log()
        fake.hipSetDevice(0)
        lib.fdkhip_plan_destroy(h)
        fake.fake_clear()
    """)


@pytest.mark.parametrize("ns,nt,na", [(4096, 4096, 2000), (2, 1, 262145), (3, 5, 1)])
def test_phantom_grid(stub, ns, nt, na):
    """The phantom's grid covers every sample and view within a grid's limits:
    less than 2^32 threads along a dimension, 65535 workgroups along y and z."""
    _run(stub, f"""
    ns, nt, na = {ns}, {nt}, {na}
    s, t, b = np.arange(ns, dtype=float), np.arange(nt, dtype=float), np.linspace(0, 6, na)
    ell = np.array([[0, 0, 0, 10, 10, 10, 0, 0, 0.5]], float)
    P = lambda a: C.c_void_p(a.ctypes.data)
    _lib.check(lib.fdkhip_ellipsoid_proj(P(s), ns, P(t), nt, P(b), None, na, 541.0, 408.0, 0.0,
                                         P(ell), 1, 1, BUF, None))
    [(dev, gx, gy, gz, threads, lds, st)] = log("launch")
    assert gx * threads >= ns * nt and gx * threads < 2 ** 32, (gx, threads)
    assert gy <= 65535 and gz <= 65535 and gy * gz * 4 >= na, (gy, gz)
    """)


@pytest.mark.parametrize("fmt", ["F32", "F16"])
@pytest.mark.parametrize("na", [24, 200])
def test_autotune_times_the_untuned_layout(stub, na, fmt):
    """The tuner times the layout of the untuned plan too, in both of its rounds:
    where that is the fastest (the only one the stand-in's clock gives 1 ms) the
    plan keeps it, slot included, and so do later plans of the geometry."""
    _run(stub, f"""
    def layout(h):
        fake.fake_clear()
        _lib.check(lib.fdkhip_plan_execute(h, BUF, BUF, BUF, None))
        cfg = (C.c_int32 * 6)()
        _lib.check(lib.fdkhip_plan_config(h, cfg))
        return list(cfg), log("launch")[-1]
    h = plan(geom(256, 256, 128, 512, 384, 0.5, 0.5, 0.8, 0.8), {na}, {fmt})
    want = layout(h)
    fake.fake_fast_lds(want[1][5])
    ms = C.c_float()
    _lib.check(lib.fdkhip_plan_autotune(h, BUF, BUF, BUF, None, 1, C.byref(ms)))
    assert ms.value == 1.0
    assert layout(h) == want
    assert layout(plan(geom(256, 256, 128, 512, 384, 0.5, 0.5, 0.8, 0.8), {na}, {fmt})) == want
    """)


def test_plan_creation_time_does_not_grow_with_slices(stub):
    """The default launch shape comes from a bounded sample of z-groups: a plan
    of 65535 slices takes no more than a few times a plan of 512 (over all groups
    it takes about 60 times as long)."""
    _run(stub, """
    def best(nz):
        t = []
        for _ in range(7):
            t0 = time.perf_counter()
            h = plan(geom(128, 128, nz, 64, 400, 4.0, 240.0 / nz, 4.0, 4.0))
            t.append(time.perf_counter() - t0)
            lib.fdkhip_plan_destroy(h)
        return min(t)
    assert best(65535) < 5 * best(512), (best(65535), best(512))
    """)


@pytest.mark.parametrize("per_scan", [False, True])
def test_batch_into_a_callers_graph(stub, per_scan):
    """A batch on a stream that the caller captures launches every scan on it, and
    neither copies, waits, nor launches a graph of its own (which would run at once,
    outside the capture), whatever calls came before; those after it go on as if it
    had not been."""
    _run(stub, f"""
    n, per_scan = 3, {per_scan}
    garr = (_lib.Geom * n)(*[geom(32 + 8 * i, 32, 24, 64, 48, 2.0, 2.0, 4.0, 4.0) for i in range(n)])
    beta = np.linspace(0, 6, 20)
    b, ba = C.c_void_p(), (C.c_void_p * n)(*[beta.ctypes.data] * n)
    _lib.check(lib.fdkhip_batch_create(C.byref(b), n, garr, (C.c_int32 * n)(20, 20, 20), ba, None, F32, 0))
    _lib.check(lib.fdkhip_batch_set_per_scan(b) if per_scan else lib.fdkhip_batch_set_config(b, 8, 16, 0))
    bufs = [(C.c_void_p * n)(*[(k + i) << 20 for i in range(n)]) for k in (1, 8)]
    S = C.c_void_p(77)
    def execute(k, direct=False):
        fake.fake_clear()
        f = lib.fdkhip_batch_execute_direct if direct else lib.fdkhip_batch_execute
        _lib.check(f(b, bufs[k], None, bufs[k], S))
        return [r[0] for r in log()]
    for warm in range(4):
        fake.fake_capturing(1)
        for k, direct in ((0, False), (1, False), (0, True), (1, True)):
            kinds = execute(k, direct)
            assert set(kinds) == {{"launch"}} and len(kinds) >= 2 * n, (warm, kinds)
        fake.fake_capturing(0)
        kinds = execute(0)
        assert ("graphlaunch" in kinds) == (warm > 0), (warm, kinds)
    """)


@pytest.mark.parametrize("ny,per_scan", [(120, False), (128, True)])
def test_batch_default_form(stub, ny, per_scan):
    """A new batch takes one launch per scan from 128 workgroups a scan in the mean
    on (64 x ny columns, one z-group: ny workgroups; one scan of 64 more and one of
    64 fewer), the work queue below."""
    _run(stub, f"""
    ys = ({ny}, {ny} + 64, {ny} - 64)
    garr = (_lib.Geom * 3)(*[geom(64, y, 16, 64, 48, 2.0, 2.0, 4.0, 4.0) for y in ys])
    beta = np.linspace(0, 6, 20)
    b, ba = C.c_void_p(), (C.c_void_p * 3)(*[beta.ctypes.data] * 3)
    for fmt in (F32, F16):
        _lib.check(lib.fdkhip_batch_create(C.byref(b), 3, garr, (C.c_int32 * 3)(20, 20, 20), ba, None,
                                           fmt, 0))
        cfg = (C.c_int32 * 6)()
        _lib.check(lib.fdkhip_batch_config(b, cfg))
        assert (cfg[0] == 0) == {per_scan} and cfg[5] == 3 * {ny}, list(cfg)
        lib.fdkhip_batch_destroy(b)
    """)
