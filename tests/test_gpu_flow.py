"""Sweeps whose workgroups wait for neighbouring batches inside one launch
(k_gs_flow), against the oracle and against the launch-by-launch sweeps, bit
for bit: one workgroup for all batches (no wait depends on another being
resident), a few, more than there are batches; small and large tiles; solves
that stop on a cap or inside a momentum iteration; two contexts at once."""
import threading
import time

import numpy as np
import pytest

import cfdl
import meshgen
from test_gpu_colour_turns import pair
from test_gpu_parity import assert_fields_equal, assert_logs_match

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wgs", ["0", "1", "3", "700"])
@pytest.mark.parametrize("edges,jitter,nsubd", [((19, 10, 13), 0.2, 4), ((35, 18, 9), 0.0, 1),
                                                ((2, 2, 2), 0.0, 1)])
def test_workgroup_counts_bitwise(monkeypatch, wgs, edges, jitter, nsubd):
    monkeypatch.setenv("CFDL_FLOW", wgs)
    eq, oc = pair(meshgen.box_mesh(*edges, jitter=jitter), nsubd)
    eq.run(1, 2, energy=True)
    oc.run(1, 2, energy=True)
    assert_fields_equal(eq, oc, ["u", "v", "w", "p", "mip", "gp", "phic", "t", "h"])
    assert_logs_match(eq.log(), oc.log())


@pytest.mark.parametrize("tile,span,nit", [("2", "3", "100"), ("16x16x4", "20", "7"),
                                           ("12", "63", "2"), ("3x5x2", "8", "11")])
def test_shapes_and_caps_bitwise(monkeypatch, tile, span, nit):
    monkeypatch.setenv("CFDL_TILE", tile)
    monkeypatch.setenv("CFDL_TILE_SPAN", span)
    eq, oc = pair(meshgen.box_mesh(14, 17, 12, jitter=0.15), 4, nit=int(nit))
    eq.run(1, 2)
    oc.run(1, 2)
    assert_fields_equal(eq, oc, ["u", "v", "w", "p", "mip", "gp", "phic"])
    assert_logs_match(eq.log(), oc.log())


def test_two_contexts_at_once():
    """Two threads, two streams: the grids share the GPU and neither waits for
    all of its workgroups to be resident."""
    mesh = cfdl.Mesh.box(40, jitter=0.1).partition(4)
    alone = cfdl.UVWP.cavity(mesh, mu=0.0025)
    alone.run(1, 3)
    want = {k: alone.get(k) for k in ("u", "p", "mip")}
    eqs = [cfdl.UVWP.cavity(mesh, mu=0.0025) for _ in range(2)]
    ts = [threading.Thread(target=eq.run, args=(1, 3)) for eq in eqs]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for eq in eqs:
        for k, v in want.items():
            assert np.array_equal(eq.get(k), v), k


def test_synchronising_an_idle_context_asks_the_device_nothing():
    """The failure word of the sweeps is read from host memory: a call that
    finds its stream idle returns without a round trip to the device (a copy
    of one word and its synchronisation take at least 8 us)."""
    eq = cfdl.UVWP.cavity(cfdl.Mesh.box(8).partition(2), mu=0.0025)
    eq.run(1, 1)
    eq.synchronize()
    best = 1.0
    for _ in range(500):
        t = time.perf_counter()
        eq.synchronize()
        best = min(best, time.perf_counter() - t)
    assert best < 4e-6, "%.1f us" % (best * 1e6)


@pytest.mark.parametrize("solve", ["uvw", "pc"])
def test_expired_wait_is_reported_until_reset(monkeypatch, solve):
    """A limit of zero lets the first wait of 1024 polls run out: a column of
    2 x 2 cells cut into 4000 batches, each waiting for the one before it (several
    us), with a workgroup for every batch.  The launch ends, every call that
    could hand out its values fails, and so do the calls after them, until a
    reset; then the context works as a new one (in an order that has no
    waits, as the limit stays)."""
    mesh = cfdl.Mesh.box(2, 2, 8000).partition(2)
    fresh = cfdl.UVWP.cavity(mesh, mu=0.0025)
    for key, value in (("FLOW_WAIT_MS", "0"), ("TILE", "2x2x2"), ("FLOW", "4000")):
        monkeypatch.setenv("CFDL_" + key, value)
    eq = cfdl.UVWP.cavity(mesh, mu=0.0025)
    if solve == "pc":
        eq.set_gs_order("colored")
        try:
            eq.run(1, 1)  # queues the sweeps; may already see that one failed
        except cfdl.CfdlError:
            pass
    else:
        with pytest.raises(cfdl.CfdlError, match="ran out of time"):
            eq.run(1, 1)
    for call in (eq.synchronize, lambda: eq.get("phic"), eq.log, eq.stats, lambda: eq.run(1, 1),
                 lambda: eq.solve("pc"), eq.solve_uvwp, lambda: eq.set_pc_order("colored")):
        with pytest.raises(cfdl.CfdlError, match="ran out of time"):
            call()
    eq.reset()
    for s in (eq, fresh):
        s.set_gs_order("colored")
        s.set_pc_order("colored")
        s.run(1, 2)
    for name in ("u", "v", "w", "p", "mip", "gp", "phic"):
        assert np.array_equal(eq.get(name), fresh.get(name)), name
    assert eq.log() == fresh.log()
    eq.set_gs_order("reference")
    with pytest.raises(cfdl.CfdlError, match="ran out of time"):
        eq.run(1, 1)  # the limit still holds
