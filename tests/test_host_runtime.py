"""Allocations that fail and routes that the host chooses, on the CPU: the
library's host code on a HIP runtime in host memory (tests/c/host_hip.c)
that fails the n-th device allocation, checks every copy against the live
ones and counts the launches.  Each test runs in
a process of its own, where that runtime is loaded first."""
import os
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def host_hip(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host_hip") / "libhost_hip.so")
    cc = os.environ.get("CC", "gcc")
    r = subprocess.run([cc, "-std=gnu11", "-Wall", "-Wextra", "-Wno-unused-parameter", "-shared", "-fPIC", "-I/opt/rocm/include", "-o", out,
                        os.path.join(ROOT, "tests", "c", "host_hip.c")], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    return out


def run(host_hip, body):
    """body after the runtime and the package are loaded: H, S, lib"""
    head = """
        import ctypes, sys
        H = ctypes.CDLL(%r, mode=ctypes.RTLD_GLOBAL)
        H.host_hip_fail.argtypes = [ctypes.c_long]
        for f in ("live", "allocs", "launches"):
            getattr(H, "host_hip_" + f).restype = ctypes.c_long
        sys.path.insert(0, %r)
        import numpy as np
        import sphradiometer_amd as S
        from sphradiometer_amd import inject
        lib = S.lib()
        assert S.gpu_available(), S.last_error()
    """ % (host_hip, ROOT)
    r = subprocess.run([sys.executable, "-c", textwrap.dedent(head) + textwrap.dedent(body)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


TD_PLAN = """
    inst = lib.instrument_array_new(0)
    for x, y, z in inject.positions("AB"):
        lib.instrument_array_append(inst, lib.instrument_new(float(x), float(y), float(z), None))
    plan = lib.correlator_network_plan_td_new(lib.correlator_network_baselines_new(inst), 1.0 / 512)
    assert plan, S.last_error()
    base = plan.contents.plans[0]
    tr, P = base.contents.transient, base.contents.power_1d.contents.l_max
    sky = lib.sh_series_new(P, 0)

    def call(n, kind):
        rng = np.random.default_rng(n)
        x = [np.ascontiguousarray(rng.standard_normal(n)) for _ in range(2)]
        nt = n - 2 * tr
        w = np.ones(nt) if kind == "flat" else rng.uniform(0.5, 1.5, nt)
        if network:
            return bool(lib.correlator_network_integrate_power_td(sky, (ctypes.c_void_p * 2)(*[v.ctypes.data for v in x]), n, (ctypes.c_void_p * 1)(w.ctypes.data), plan))
        s = lib.correlator_baseline_integrate_power_td(x[1].ctypes.data, x[0].ctypes.data, w.ctypes.data, n, base)
        ok = bool(s)
        if ok:
            lib.sh_series_free(s)
        return ok

"""

TD_GROWTH = """
    small, n = 2 * tr + 500, 2 * tr + 500
    assert call(small, "flat") and call(small, "random")
    failed = 0
    # every growth of every call fails once; the smaller calls after it run
    # in whole buffers, and so does the larger one when memory is there
    for kind in ("flat", "random"):
        for k in range(1, 12):
            n = 2 * n
            H.host_hip_fail(k)
            ok = call(n, kind)
            H.host_hip_fail(0)
            failed += not ok
            assert call(small, "flat") and call(small, "random"), (kind, k)
            assert call(n, kind), (kind, k)
            n = n if n < 400000 else small
            if n == small:
                lib.correlator_network_plan_td_free(plan)
                plan = lib.correlator_network_plan_td_new(lib.correlator_network_baselines_new(inst), 1.0 / 512)
                base = plan.contents.plans[0]
                assert call(small, "flat") and call(small, "random")
    print("failed", failed)
"""


@pytest.mark.parametrize("network", [False, True])
def test_td_buffers_after_a_failed_growth(host_hip, network):
    """a growth that fails leaves no capacity behind for the buffer it
    freed: later calls that fit the old capacity allocate again"""
    out = run(host_hip, "    network = %r\n" % network + TD_PLAN + TD_GROWTH)
    assert int(out.split()[-1]) >= 4, out


@pytest.mark.parametrize("network", [False, True])
def test_td_without_pinned_memory(host_hip, network):
    """without pinned memory the copies are made directly, and the calls
    succeed, the first and those after it"""
    run(host_hip, "    network = %r\n" % network + TD_PLAN + """
    for on in (1, 0, 1):
        H.host_hip_fail_pinned(on)
        for n in (2 * tr + 3000 * (1 + on), 2 * tr + 400):
            assert call(n, "flat") and call(n, "random"), (on, n, S.last_error())
""")


def test_td_flat_window_route(host_hip):
    """windows with at most half as many differences as samples take the
    flat-window route (two launches more), whatever the differences are:
    at the limit and past it, in blocks of 64 and their remainders, NaN and
    infinities (their differences are not zero), zeros of either sign (are)"""
    run(host_hip, "    network = False\n" + TD_PLAN + """
    def flat(w):
        x = np.ones(len(w) + 2 * tr)
        n0 = H.host_hip_launches()
        s = lib.correlator_baseline_integrate_power_td(x.ctypes.data, x.ctypes.data, w.ctypes.data, len(x), base)
        assert s, S.last_error()
        lib.sh_series_free(s)
        n = H.host_hip_launches() - n0
        assert n in (4, 6), n
        return n == 6

    def count(w):
        with np.errstate(invalid="ignore"):
            return int(np.sum(w[:-1] - w[1:] != 0.0)) + (w[0] != 0.0) + (w[-1] != 0.0)

    rng = np.random.default_rng(1)
    limit = 0
    for nt in (2, 3, 63, 64, 65, 66, 128, 129, 130, 301, 640):
        for trial in range(60):
            w = np.full(nt, rng.choice([0.0, 1.0]))
            k = int(rng.integers(0, nt // 2 + 2))
            at = rng.choice(nt, min(k, nt), replace=False)
            w[at] = rng.choice([0.0, -0.0, 1.0, 2.0, np.nan, np.inf, 1e-310], len(at))
            if trial % 3 == 0:	# exactly the limit, or one past it
                w = np.zeros(nt)
                w[np.sort(rng.choice(nt, max(1, nt // 4), replace=False))] = rng.uniform(1, 2, max(1, nt // 4))
                while count(w) < nt // 2 + trial % 2 and (w == 0.0).any():
                    z = np.flatnonzero(w == 0.0)
                    w[z[rng.integers(len(z))]] = rng.uniform(1, 2)
            limit += count(w) == nt // 2
            assert flat(w) == (count(w) <= nt // 2), (nt, trial, count(w))
    assert limit > 20, limit
    """)


def test_device_alloc_after_a_failure(host_hip):
    """an allocation that failed is reported once, by the call that asked"""
    run(host_hip, """
    H.host_hip_fail(1)
    try:
        S.DeviceBuffer(100)
        raise SystemExit("no error")
    except RuntimeError:
        pass
    x = np.zeros(100)
    H.host_hip_fail(1)
    f = None
    try:
        f = S.tseries_to_fseries(x)
    except RuntimeError:
        pass
    a = S.DeviceBuffer.from_numpy(np.zeros(50, dtype=np.complex128))
    h = S.Healpix(4, 4, S.FP64)
    m = S.DeviceBuffer(h.npix * 8)
    h.maps(a.ptr, 1, m.ptr)
    H.host_hip_fail(1)
    try:
        S.DeviceBuffer(100)
    except RuntimeError:
        pass
    h.maps(a.ptr, 1, m.ptr)
""")


def test_healpix_without_memory_for_tables(host_hip):
    """the tables of the maps are optional: without memory for them the plan
    runs the per-ring form; without memory for the coefficients there is no
    plan; nothing is left allocated"""
    run(host_hip, """
    for prec in (S.FP64, S.MIXED):
        start = H.host_hip_live()
        n0 = H.host_hip_allocs()
        h = S.Healpix(50, 32, prec)
        n = H.host_hip_allocs() - n0
        assert h.form(1000) == 1 and n == 4, n
        del h
        for k in range(1, n + 1):
            H.host_hip_fail(k)
            try:
                h = S.Healpix(50, 32, prec)
            except RuntimeError:
                h = None
            H.host_hip_fail(0)
            assert (h is None) == (k == 1), k
            if h:
                assert h.form(1000) == 0
                a, m = S.DeviceBuffer(51 ** 2 * 16), S.DeviceBuffer(h.npix * 8)
                h.maps(a.ptr, 1, m.ptr)
                a.free(), m.free()
                del h
            assert H.host_hip_live() == start, k
    """)


def test_one_map_makes_no_tables(host_hip, tmp_path):
    """to a file and from healpy coefficients: a plan used for one series holds the coefficients alone"""
    run(host_hip, """
    s = S.series_from_numpy(np.ones(33 ** 2), 32, 0)
    start, n0 = H.host_hip_live(), H.host_hip_allocs()
    assert lib.sh_series_write_healpix_map(s, %r) == 0, S.last_error()
    assert H.host_hip_allocs() - n0 == 3 and H.host_hip_live() == start
    from sphradiometer_amd import healpix
    n0 = H.host_hip_allocs()
    healpix.healpy_alm_to_map(np.ones(healpix.healpy_alm_length(32, 32)), 32, 32)
    assert H.host_hip_allocs() - n0 == 3
    """ % os.path.join(str(tmp_path), "map.fits").encode())
