"""The V-cycle's levels in colour numbering against the oracle's, bit for bit:
level 0 of two and of three colours, coarse levels of many colours whose last
ones share a workgroup, rows longer than one load group, hierarchies of one
level, of workgroup-only levels and of several grid-wide ones, in FP64 and
with the FP32 V-cycle."""
import numpy as np
import pytest

import meshgen
from test_gpu_colour_turns import pair, three_blocks
from test_gpu_parity import assert_fields_equal, assert_logs_match

MESHES = {
    "one level": lambda: meshgen.box_mesh(4, 3, 5),
    "one cell": lambda: meshgen.box_mesh(1),
    "65 cells": lambda: meshgen.box_mesh(13, 5, 1, jitter=0.2),
    "workgroup levels": lambda: meshgen.box_mesh(9, 11, 13, jitter=0.2),
    "even box": lambda: meshgen.box_mesh(32, 32, 16),
    "odd box": lambda: meshgen.box_mesh(47, 41, 37, jitter=0.2),
    "three blocks": lambda: three_blocks(13, 22),
    "thin": lambda: meshgen.box_mesh(150, 70, 1),
}


@pytest.mark.gpu
@pytest.mark.parametrize("order", ["mgcg", "mgcg-mixed"])
@pytest.mark.parametrize("mesh", list(MESHES))
def test_levels_bitwise(mesh, order):
    eq, oc = pair(MESHES[mesh](), 1, dt=float("inf"))
    for s in (eq, oc):
        s.set_relaxation(0.7, 0.3)
        s.set_pc_order(order)
        s.set_gs_order("colored")
    eq.run(1, 2)
    oc.run(1, 2)
    assert_fields_equal(eq, oc, ["u", "v", "w", "p", "mip", "gp", "phic"])
    assert_logs_match(eq.log(), oc.log())


@pytest.mark.gpu
def test_non_finite_coefficients_end_the_solve():
    """A forward sweep starts without reading its first colour's rows; a
    coefficient that is not finite still keeps the solve from starting."""
    eq, oc = pair(meshgen.box_mesh(8), 1)
    for s in (eq, oc):
        s.set_pc_order("mgcg")
    eq.run(1, 1)
    for bad in (np.inf, -np.inf, np.nan):
        eq.calc_coef_p()
        anb = eq.get("anb")
        anb[100] = bad
        eq.set("anb", anb)
        eq.set_a_0("phic")
        eq.clear_log()
        eq.solve("pc")
        assert eq.log()[0][1] == 0
        assert not eq.get("phic").any()
