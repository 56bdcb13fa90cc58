"""pz_get_ddr_noalloc against pz_get_ddr, bit for bit, over the numbers of
columns that a workgroup takes (one, two, four, with a short last group and
with tiles that do not divide by the eight chiplets), register, Stockham and
direct-sum transform lengths; written over its own input; and two handles of
one process at once, whose results must not depend on each other."""
import ctypes

import numpy as np
import pytest

from test_zz_no_alloc import _Device, _hip

pytestmark = pytest.mark.gpu


def _run(n_r):
    from pizza_amd.config import default_config
    from pizza_amd.runtime import Run
    return Run(default_config(n_r_max=n_r, n_cheb_max=n_r, m_max=6, radratio=0.35, cheb_method="colloc",
                              matrix_solve="direct"))


def _field(rng, n_m, n_r):
    return rng.standard_normal((n_m, n_r)) + 1j * rng.standard_normal((n_m, n_r))


def _call(run, d_f, d_1, d_2, n_m, dct):
    from pizza_amd.runtime import lib
    rc = lib().pz_get_ddr_noalloc(run.h, d_f.ptr, d_1.ptr, d_2.ptr if d_2 is not None else None, n_m, dct)
    assert rc == 0, lib().pz_last_error(run.h)


@pytest.mark.parametrize("n_r,n_m,dct,second", [
    (33, 1, 1, True), (33, 1025, 1, True), (33, 1030, 0, False), (65, 513, 1, True), (80, 515, 1, True), (97, 1027, 1, False),
    (193, 1358, 1, True), (193, 511, 0, True), (257, 520, 1, True)])
def test_noalloc_columns(n_r, n_m, dct, second):
    print(f"case: noalloc derivative n_r {n_r}, {n_m} columns", flush=True)
    if n_r < 257:
        run = _run(n_r)
    else:  # the longest grid belongs to finite differences
        from pizza_amd import workloads as W
        from pizza_amd.runtime import Run
        run = Run(W.c5_fd(n_r=257, m_max=6))
    hip, f = _hip(), _field(np.random.default_rng(5), n_m, n_r)
    want = run.get_ddr(f, bool(dct)) if second else (run.get_dr(f, bool(dct)),)
    x, o1, o2 = (_Device(hip, n_m * n_r) for _ in range(3))
    x.put(f.T)
    assert hip.hipDeviceSynchronize() == 0
    _call(run, x, o1, o2 if second else None, n_m, dct)
    assert hip.hipDeviceSynchronize() == 0
    for o, w in zip((o1, o2), want):
        assert np.array_equal(o.get((n_r, n_m)).T, w)
    _call(run, x, x, o2 if second else None, n_m, dct)  # in place
    assert hip.hipDeviceSynchronize() == 0
    assert np.array_equal(x.get((n_r, n_m)).T, want[0])
    for b in (x, o1, o2):
        b.free()


def test_noalloc_two_handles_at_once():
    print("case: noalloc derivative, two handles", flush=True)
    hip, rng = _hip(), np.random.default_rng(6)
    runs, fs = [_run(97), _run(193)], [_field(rng, 2000, 97), _field(rng, 1300, 193)]
    want = [r.get_ddr(f, True) for r, f in zip(runs, fs)]
    bufs = [[_Device(hip, f.size) for _ in range(3)] for f in fs]
    for b, f in zip(bufs, fs):
        b[0].put(f.T)
    assert hip.hipDeviceSynchronize() == 0
    for _ in range(20):
        for r, f, b in zip(runs, fs, bufs):
            _call(r, b[0], b[1], b[2], f.shape[0], 1)
    assert hip.hipDeviceSynchronize() == 0
    for b, f, w in zip(bufs, fs, want):
        for o, v in zip(b[1:], w):
            assert np.array_equal(o.get(f.T.shape).T, v)
        for d in b:
            d.free()


@pytest.mark.parametrize("n_r,n_m,at", [(97, 1027, (0, 5, 11)), (33, 700, (700, 0, 33)), (65, 513, (3, 3, 0)), (33, 64, (0, 2112, 31))])
def test_noalloc_arrays_that_overlap_in_part(n_r, n_m, at):
    """f, df and ddf at offsets of one buffer, each array overlapping the next
    in part (or, where offsets are equal, wholly): the derivatives are those
    of f as it was before the call, ddf written after df."""
    print(f"case: noalloc derivative, overlapping arrays, n_r {n_r}, {n_m} columns", flush=True)
    run, hip, S = _run(n_r), _hip(), n_m * n_r
    f = _field(np.random.default_rng(8), n_m, n_r)
    buf = _Device(hip, S + max(at))
    host = np.zeros(S + max(at), dtype=np.complex128)
    host[at[0]:at[0] + S] = f.T.ravel()
    buf.put(host)
    want = host.copy()
    d1, d2 = run.get_ddr(f, True)
    want[at[1]:at[1] + S] = d1.T.ravel()
    want[at[2]:at[2] + S] = d2.T.ravel()
    assert hip.hipDeviceSynchronize() == 0

    class _At:
        def __init__(self, o):
            self.ptr = ctypes.c_void_p(buf.ptr.value + 16 * o)

    _call(run, _At(at[0]), _At(at[1]), _At(at[2]), n_m, 1)
    assert hip.hipDeviceSynchronize() == 0
    assert np.array_equal(buf.get(want.shape), want)
    buf.free()


@pytest.mark.parametrize("at", [(0, 4000, 8000), (0, 5, 11)])
def test_noalloc_under_capture(at):
    """The call captured on the handle's stream and replayed with other inputs,
    eager work between the replays: arrays apart (one kernel) and arrays that
    overlap in part (temporaries, copies)."""
    print(f"case: noalloc derivative captured, offsets {at}", flush=True)
    n_r, n_m = 33, 100
    run, hip, S = _run(n_r), _hip(), n_m * n_r
    stream = ctypes.c_void_p(run.stream())
    buf, rng = _Device(hip, S + max(at)), np.random.default_rng(9)

    class _At:
        def __init__(self, o):
            self.ptr = ctypes.c_void_p(buf.ptr.value + 16 * o)

    graph, ex = ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamBeginCapture(stream, 1) == 0  # thread-local
    _call(run, _At(at[0]), _At(at[1]), _At(at[2]), n_m, 1)
    assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)) == 0
    for _ in range(4):
        f = _field(rng, n_m, n_r)
        host = np.zeros(S + max(at), dtype=np.complex128)
        host[at[0]:at[0] + S] = f.T.ravel()
        want = host.copy()
        d1, d2 = run.get_ddr(f, True)  # eager work of the same handle
        want[at[1]:at[1] + S] = d1.T.ravel()
        want[at[2]:at[2] + S] = d2.T.ravel()
        buf.put(host)
        assert hip.hipDeviceSynchronize() == 0
        assert hip.hipGraphLaunch(ex, stream) == 0
        assert hip.hipDeviceSynchronize() == 0
        assert np.array_equal(buf.get(want.shape), want)
    assert hip.hipGraphExecDestroy(ex) == 0 and hip.hipGraphDestroy(graph) == 0
    buf.free()
