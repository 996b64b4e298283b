"""Large host transfers through the pinned slots: lengths around the shortest
one that takes them, with and without a last partial chunk, against the
runtime's own copy (pinned host memory takes that), before and after the slots
are given back, and from several threads.  All copies are exact."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 192 V and 576 V bytes around 8 MiB; three 4 MiB chunks exactly; many
SIZES = [(10, 12, 19, 19), (16, 16, 16, 11), (4, 16, 32, 32), (20, 18, 22, 14), (32, 16, 16, 16)]


def _ptr(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


@pytest.fixture
def pinned():
    """pinned(n): n doubles of pinned host memory, freed after the test."""
    hip = ctypes.CDLL("libamdhip64.so")
    blocks = []

    def get(n):
        p = ctypes.c_void_p()
        assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(8 * n), ctypes.c_uint(0)) == 0
        blocks.append(p)
        return np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_double)), shape=(n,))

    yield get
    for p in blocks:
        hip.hipHostFree(p)


def _round(Q, pinned, f, n, pageable_up, seed, fn):
    rng = np.random.default_rng(seed)
    src = rng.standard_normal(n)
    out = pinned(n) if pageable_up else np.zeros(n)
    if not pageable_up:
        p = pinned(n)
        p[:] = src
    up, down = fn
    lib = Q.lib()
    assert up(lib, f, _ptr(src if pageable_up else p)) == 0
    assert down(lib, f, _ptr(out)) == 0
    assert np.array_equal(out, src)


SPINOR = (lambda lib, f, p: lib.qcd_hip_spinor_upload(f.h, 0, p),
          lambda lib, f, p: lib.qcd_hip_spinor_download(f.h, 0, p))
GAUGE = (lambda lib, f, p: lib.qcd_hip_gauge_upload(f.h, p), lambda lib, f, p: lib.qcd_hip_gauge_download(f.h, p))
PROP = (lambda lib, f, p: lib.qcd_hip_propagator_upload(f.h, 0, p),
        lambda lib, f, p: lib.qcd_hip_propagator_download(f.h, 0, p))


@pytest.mark.parametrize("L", SIZES)
def test_pageable_against_pinned(gpu, pinned, L):
    Q = gpu
    lat, V = Q.Lattice(L), int(np.prod(L))
    cases = [(Q.Spinor(lat), 24 * V, SPINOR), (Q.Gauge(lat), 72 * V, GAUGE)]
    if V <= 50000:
        cases.append((Q.Spinor(lat, nrhs=12), 288 * V, PROP))
    for f, n, fn in cases:
        _round(Q, pinned, f, n, True, 1, fn)
        _round(Q, pinned, f, n, False, 2, fn)
        Q.lib().qcd_hip_release_cache()
        _round(Q, pinned, f, n, True, 3, fn)


def test_transfers_from_several_threads(gpu):
    Q = gpu
    L = (20, 18, 22, 14)
    lat, V = Q.Lattice(L), int(np.prod(L))
    bad = []

    def work(i):
        f = Q.Spinor(lat)
        src = np.random.default_rng(i).standard_normal(24 * V)
        out = np.zeros(24 * V)
        for _ in range(3):
            if SPINOR[0](Q.lib(), f, _ptr(src)) or SPINOR[1](Q.lib(), f, _ptr(out)):
                bad.append(i)
        if not np.array_equal(out, src):
            bad.append(i)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad
