"""Sweeps whose workgroups wait for neighbouring batches inside one launch
(k_gs_flow), against the oracle and against the launch-by-launch sweeps, bit
for bit: one workgroup for all batches (no wait depends on another being
resident), a few, more than there are batches; small and large tiles; solves
that stop on a cap or inside a momentum iteration; two contexts at once."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

import cfdl
import meshgen
import oracle_lib
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


def shuffled_pair(n, seed, shuffle):
    """A box whose cells are numbered at random, and its oracle; with shuffle
    the context is given the cells' centres in another order, so that a
    sweep's tiles are groups of cells from all over the mesh."""
    g = meshgen.box_mesh(n)
    rng = np.random.default_rng(seed)
    ne = g["ne"]
    cells = np.array(g["e2vx"]).reshape(-1, 8)
    cells[:ne] = cells[:ne][rng.permutation(ne)]
    g["e2vx"] = cells.reshape(-1)
    m = cfdl.Mesh.from_elements(g["x"], g["y"], g["z"], g["etype"], g["esec"], g["e2vx"],
                                names=g["names"]).partition(2)
    i, bc = m.info(), meshgen.cavity_bc(g)
    oc = oracle_lib.OracleCase(g, bc, nsubd=2)
    xyz = [m.get(k) for k in ("xc", "yc", "zc")]
    order = rng.permutation(ne)
    if shuffle:
        for a in xyz:
            a[:ne] = a[:ne][order]
    eq = cfdl.UVWP.from_arrays(
        i["ne"], i["nf"], i["nbf"], *[m.get(k) for k in ("ef2nb_idx", "ef2nb", "s2g", "bs")], *xyz,
        *[m.get(k) for k in ("vol", "aip", "rip", "esec")], bc, 2,
        *[m.get(k) for k in ("gf2g", "g2gf", "g2gf_idx")], np.ones(ne), np.full(ne, 0.01), 0.01)
    return eq, oc, rng


@pytest.mark.parametrize("shuffle", [False, True])
def test_batches_with_many_neighbours_run_step_by_step(shuffle):
    """The waiting wavefront has a lane per neighbouring batch: a schedule
    with 64 or more on one side (random tiles: up to 127 for u, v, w and 99
    in the pc system, in segments of at most 54 cells) runs a launch a step,
    without being told to; the same cells in tiles of neighbours run in one
    launch an iteration or block.  Both give the oracle's bits."""
    with pytest.MonkeyPatch.context() as mp:
        mp.setenv("CFDL_TILE", "1" if shuffle else "4")
        eq, oc, rng = shuffled_pair(13, 3, shuffle)
    ne, idx = oc.c.ne, oc.arr("ef2nb_idx") - 1
    anb = rng.uniform(0.5, 1.0, idx[-1])
    ap = np.add.reduceat(anb, idx[:-1]) + 0.5
    for s in (eq, oc):
        put = eq.set if s is eq else lambda k, v: oc.arr(k).__setitem__(slice(None), v)
        put("anb", anb)
        put("ap", ap)
    rhs = {k: rng.uniform(-1.0, 1.0, ne) for k in ("bu", "bv", "bw", "b")}
    for k, v in rhs.items():
        eq.set(k, v)
        oc.arr(k)[:] = v
    for k in ("u", "v", "w", "phic"):
        eq.set_a_0(k)
        oc.arr(k)[:] = 0.0
    eq.solve_gs_uvw()
    momentum = eq.stats()["gs_launches"]
    iterations = max(line[1] for line in eq.log())
    eq.reset_stats()
    eq.solve("pc")
    pc = eq.stats()["pc_launches"]
    assert iterations >= 2
    assert (momentum > 2 * iterations and pc > 100) if shuffle else (momentum == iterations and pc == 50)
    L, c = oracle_lib.lib(), oc.c
    L.or_solve_gs.argtypes = [C.POINTER(oracle_lib.OrCase), C.c_char_p, oracle_lib.PD, oracle_lib.PD,
                              oracle_lib.PD, oracle_lib.PD, oracle_lib.PI, oracle_lib.PI,
                              C.c_int, C.c_int, C.c_int, C.c_int]
    for phi, b in (("u", "bu"), ("v", "bv"), ("w", "bw")):
        L.or_solve_gs(oc.p, phi.encode(), getattr(c, phi), c.ap, c.anb, getattr(c, b),
                      c.ef2nb_idx, c.ef2nb, c.ne, c.nf, c.nbf, c.nit)
    L.or_solve(oc.p, b"pc", c.phic)
    assert_fields_equal(eq, oc, ["u", "v", "w", "phic"])


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
