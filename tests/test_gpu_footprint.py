"""Device memory of a serving context: within the figure that admission counts
with, in both assembly precisions, and the same after changing precision."""
import ctypes as C

import numpy as np
import pytest

import cfdl
from cfdl import serving


def test_admitted_figure():
    """64 MiB and 1,344 B a cell: a budget keeps admitting as many contexts."""
    assert serving.footprint(96) == (64 << 20) + 1344 * 96 ** 3


def free_bytes():
    h = C.CDLL("libamdhip64.so.7")  # the soname the library loaded
    free, total = C.c_size_t(), C.c_size_t()
    assert h.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n,bits", [("cavity", 16, 32), ("channel", 48, 32), ("cavity", 64, 64),
                                         ("channel", 96, 32), ("cavity", 96, 64),
                                         ("cavity", 112, 32), ("cavity", 128, 32),
                                         ("cavity", 128, 64)])
def test_contexts_fit_their_footprint(kind, n, bits):
    pool = serving.ContextPool(assembly_bits=bits)
    first = pool.acquire(kind, n, 1e15)  # modules and shared buffers load once
    first[1].run(1, 1)
    first[1].synchronize()
    before, count = free_bytes(), 3
    for _ in range(count):
        pool.acquire(kind, n, 1e15)[1].run(1, 1)
    used = (before - free_bytes()) / count
    pool.close()
    assert used <= serving.footprint(n), "%.0f B a cell" % ((used - (64 << 20)) / n ** 3)


@pytest.mark.gpu
def test_precision_changes_keep_the_results():
    """FP64, FP32 and FP64 again on one context, each like a fresh one."""
    mesh = cfdl.Mesh.box(12, 9, 7, jitter=0.2).partition(1)

    def make():
        eq = cfdl.UVWP.cavity(mesh, mu=0.0025, dt=float("inf"))
        eq.set_relaxation(0.7, 0.3)
        eq.set_gs_order("colored")
        eq.set_pc_order("mgcg")
        return eq

    eq = make()
    for bits in (64, 32, 32, 64, 32):
        eq.set_assembly_precision(bits)
        eq.reset()
        eq.run(1, 2)
        fresh = make()
        fresh.set_assembly_precision(bits)
        fresh.run(1, 2)
        for name in ("u", "v", "w", "p", "mip", "ap", "anb", "bu", "dc"):
            assert np.array_equal(eq.get(name), fresh.get(name)), (bits, name)
