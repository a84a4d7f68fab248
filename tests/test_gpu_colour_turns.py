"""Colour orders whose turning colours share a launch, bit for bit against the
oracle's sequential sweeps: boxes (two colours) and three hexahedral blocks
around an edge, whose cell graph has odd cycles (three colours, where a
symmetric pair is 1 2 33 2 1 and the turn between two pairs another double)."""
import numpy as np
import pytest

import cfdl
import meshgen
import oracle_lib
from test_gpu_parity import assert_fields_equal, assert_logs_match

NAMES = ["cells", "bottom", "side", "top"]


def three_blocks(m, layers):
    """A triangle cut into three quadrilaterals at its centroid, each m x m,
    extruded: hexahedra, sections bottom, side and top."""
    c = [np.array(q) for q in ((0.0, 0.0), (1.0, 0.1), (0.4, 0.9))]
    mid = [(c[i] + c[(i + 1) % 3]) / 2 for i in range(3)]
    g = sum(c) / 3
    ids, pts = {}, []

    def vid(q):
        key = (round(q[0], 9), round(q[1], 9))
        if key not in ids:
            ids[key] = len(pts)
            pts.append(q)
        return ids[key]

    quads = []
    for i in range(3):
        a, b, d, e = c[i], mid[i], g, mid[i - 1]
        grid = [[vid((1 - s) * (1 - t) * a + s * (1 - t) * b + s * t * d + (1 - s) * t * e)
                 for s in np.linspace(0, 1, m + 1)] for t in np.linspace(0, 1, m + 1)]
        quads += [(grid[t][s], grid[t][s + 1], grid[t + 1][s + 1], grid[t + 1][s])
                  for t in range(m) for s in range(m)]
    n2 = len(pts)
    xy = np.array(pts)
    x, y = np.tile(xy[:, 0], layers + 1), np.tile(xy[:, 1], layers + 1)
    z = np.repeat(np.linspace(0.0, 0.8, layers + 1), n2)
    cells = [[1 + v + n2 * k for v in q] + [1 + v + n2 * (k + 1) for v in q]
             for k in range(layers) for q in quads]
    edges = {}
    for q in quads:
        for i in range(4):
            edges.setdefault(frozenset((q[i], q[(i + 1) % 4])), []).append((q[i], q[(i + 1) % 4]))
    rim = [e[0] for e in edges.values() if len(e) == 1]
    bottom = [[1 + q[0], 1 + q[3], 1 + q[2], 1 + q[1]] for q in quads]
    side = [[1 + a + n2 * k, 1 + b + n2 * k, 1 + b + n2 * (k + 1), 1 + a + n2 * (k + 1)]
            for k in range(layers) for a, b in rim]
    top = [[1 + v + n2 * layers for v in q] for q in quads]
    e2vx, esec, at = [r for r in cells], [(1, len(cells))], len(cells)
    for sec in (bottom, side, top):
        e2vx += [r + [0] * 4 for r in sec]
        esec.append((at + 1, at + len(sec)))
        at += len(sec)
    return dict(nvx=len(x), x=x, y=y, z=z, e2vx=np.array(e2vx, np.int32).reshape(-1),
                etype=np.array([17, 7, 7, 7], np.int32), esec=np.array(esec, np.int32).reshape(-1),
                names=NAMES, ne=len(cells), nbf=at - len(cells))


def pair(g, nsubd, **kw):
    mesh = cfdl.Mesh.from_elements(g["x"], g["y"], g["z"], g["etype"], g["esec"], g["e2vx"],
                                   names=g["names"]).partition(nsubd)
    eq = cfdl.UVWP.cavity(mesh, mu=0.0025, **kw)
    oc = oracle_lib.OracleCase(g, meshgen.cavity_bc(g), nsubd=nsubd, mu=0.0025, **kw)
    return eq, oc


def colours(g, order):
    """Greedy colours of the cell graph, from the vertices the cells share."""
    face = {}
    e = g["e2vx"].reshape(-1, 8)[:g["ne"]]
    for i, v in enumerate(e):
        for f in ((0, 1, 2, 3), (4, 5, 6, 7), (0, 1, 5, 4), (1, 2, 6, 5), (2, 3, 7, 6), (3, 0, 4, 7)):
            face.setdefault(frozenset(v[list(f)].tolist()), []).append(i)
    near = [[] for _ in e]
    for p in face.values():
        if len(p) == 2:
            near[p[0]].append(p[1])
            near[p[1]].append(p[0])
    col = {}
    for i in order:
        used = {col[j] for j in near[i] if j in col}
        col[i] = next(q for q in range(9) if q not in used)
    return max(col.values()) + 1


def test_three_blocks_need_three_colours():
    g = three_blocks(3, 4)
    assert colours(g, range(g["ne"])) >= 3
    b = meshgen.box_mesh(5)
    assert colours(b, range(b["ne"])) == 2


@pytest.mark.gpu
@pytest.mark.parametrize("m,layers", [(1, 1), (2, 3), (5, 6)])
@pytest.mark.parametrize("order,nsubd", [("colored", 1), ("colored", 4), ("mixed", 2)])
def test_three_blocks_bitwise(m, layers, order, nsubd):
    if m == 1:
        nsubd = 1
    g = three_blocks(m, layers)
    eq, oc = pair(g, nsubd)
    for s in (eq, oc):
        if nsubd > 1:  # one subdomain: the pc solve is solve_gs
            s.set_pc_order(order)
        s.set_gs_order("colored")
    eq.run(2, 2)
    oc.run(2, 2)
    assert_fields_equal(eq, oc, ["u", "v", "w", "p", "mip", "gp", "phic"])
    assert_logs_match(eq.log(), oc.log())


@pytest.mark.gpu
@pytest.mark.parametrize("nit", [1, 2, 7, 100])
@pytest.mark.parametrize("order", ["colored", "mixed"])
def test_block_caps_bitwise(nit, order):
    """The iteration cap ends a solve after any block."""
    g = meshgen.box_mesh(9, 7, 5, jitter=0.2)
    eq, oc = pair(g, 4, nit=nit)
    for s in (eq, oc):
        s.set_pc_order(order)
        s.set_gs_order("colored")
    eq.run(1, 2)
    oc.run(1, 2)
    assert_fields_equal(eq, oc, ["u", "v", "w", "p", "mip", "gp", "phic"])
    assert_logs_match(eq.log(), oc.log())
