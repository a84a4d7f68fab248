"""Reading fields back: copies of one piece and of several, to the last byte,
into pageable and pinned memory, and a pinned destination's speed."""
import ctypes as C
import time

import numpy as np
import pytest

import cfdl

pytestmark = pytest.mark.gpu

PD = C.POINTER(C.c_double)


def read(eq, name, ptr):
    n, fid = eq.sizes[name], cfdl.solver.FIELDS[name]
    assert cfdl.load_library().cfdl_get_field(eq._h, fid, C.cast(ptr, PD), n) == 0


@pytest.fixture
def hip():
    """Pinned host memory and copies by the HIP runtime the library uses."""
    cfdl.load_library()
    h = C.CDLL("libamdhip64.so.7")  # the soname the library loaded
    h.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    h.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    h.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    h.hipHostFree.argtypes = h.hipFree.argtypes = [C.c_void_p]
    live = []

    def pinned(n):
        p = C.c_void_p()
        assert h.hipHostMalloc(C.byref(p), 8 * n, 0) == 0
        live.append((h.hipHostFree, p))
        return np.ctypeslib.as_array(C.cast(p, PD), (n,))

    def device(n):
        p = C.c_void_p()
        assert h.hipMalloc(C.byref(p), 8 * n) == 0
        live.append((h.hipFree, p))
        return p

    h.pinned, h.device = pinned, device
    yield h
    for free, p in live:
        free(p)


# cells * 8 bytes around one, two and three pieces of 2 MiB
@pytest.mark.parametrize("edges", [(2, 3, 5), (64, 64, 64), (65, 64, 64), (64, 64, 128),
                                   (64, 128, 65), (96, 96, 86)])
def test_every_size_into_pageable_and_pinned_memory(hip, edges):
    eq = cfdl.UVWP.cavity(cfdl.Mesh.box(*edges).partition(1), mu=0.01)
    for name in ("ap", "u"):
        want = np.random.default_rng(5).standard_normal(eq.sizes[name])
        eq.set(name, want)
        assert np.array_equal(eq.get(name), want)
        p = hip.pinned(want.size)
        read(eq, name, p.ctypes.data)
        assert np.array_equal(p, want)
        shifted = np.full(want.size + 2, np.nan)  # not at the start of its pages
        read(eq, name, shifted.ctypes.data + 8)
        assert np.array_equal(shifted[1:-1], want) and np.isnan(shifted[[0, -1]]).all()
    eq.close()


def test_a_pinned_destination_takes_one_copy(hip):
    """As fast as hipMemcpy of the same bytes to the same place (staged through
    the CPU it took twice as long)."""
    eq = cfdl.UVWP.cavity(cfdl.Mesh.box(96).partition(1), mu=0.01)
    n = eq.sizes["gu"]
    p, d = hip.pinned(n), hip.device(n)

    def best(call):
        t = []
        for _ in range(10):
            s = time.perf_counter()
            call()
            t.append(time.perf_counter() - s)
        return min(t)

    direct = best(lambda: hip.hipMemcpy(p.ctypes.data, d, 8 * n, 2))
    assert best(lambda: read(eq, "gu", p.ctypes.data)) < 1.4 * direct
    eq.close()
