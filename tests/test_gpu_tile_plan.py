"""The tile shape and layer-aligned cuts the sweep schedules are planned with,
against the oracle bit for bit: uneven and one-layer boxes, distorted cells,
more layers than a tile holds, edges one past a tile's, a mesh whose layers
are no planes (three blocks around an edge); the host memory planning takes."""
import os
import subprocess
import sys

import numpy as np
import pytest

import cfdl
import meshgen
from test_gpu_colour_turns import pair, three_blocks
from test_gpu_parity import assert_fields_equal, assert_logs_match

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("edges,jitter,nsubd", [
    ((5, 1, 1), 0.0, 1), ((1, 7, 3), 0.1, 1), ((33, 9, 6), 0.2, 2), ((17, 17, 17), 0.2, 4),
    ((9, 17, 5), 0.0, 4), ((40, 8, 12), 0.15, 8), ((4, 4, 49), 0.2, 1), ((13, 24, 9), 0.2, 1)])
def test_boxes_bitwise(edges, jitter, nsubd):
    eq, oc = pair(meshgen.box_mesh(*edges, jitter=jitter), nsubd)
    eq.run(1, 2)
    oc.run(1, 2)
    assert_fields_equal(eq, oc)
    assert_logs_match(eq.log(), oc.log())


@pytest.mark.parametrize("nsubd", [1, 3])
def test_three_blocks_bitwise(nsubd):
    eq, oc = pair(three_blocks(6, 9), nsubd)
    eq.run(1, 2)
    oc.run(1, 2)
    assert_fields_equal(eq, oc)
    assert_logs_match(eq.log(), oc.log())


def graded(n, s):
    """A box whose cells grow by a factor e^s along each axis."""
    g = meshgen.box_mesh(n)
    for k in ("x", "y", "z"):
        top = g[k].max()
        g[k] = top * (np.exp(s * g[k] / top) - 1.0) / (np.exp(s) - 1.0)
    return g


@pytest.mark.parametrize("n,s,nsubd", [(24, 2.0, 4), (24, 2.0, 2), (15, 4.0, 4), (20, 3.0, 1)])
def test_graded_boxes_bitwise(n, s, nsubd):
    """Cells much finer than the mean: the boxes of the usual shapes hold too
    many of them for the LDS or the walk, and finer shapes take their place,
    so that the sweeps of a block still run in one launch."""
    eq, oc = pair(graded(n, s), nsubd)
    eq.run(1, 2)
    oc.run(1, 2)
    assert_fields_equal(eq, oc)
    assert_logs_match(eq.log(), oc.log())
    st = eq.stats()
    if nsubd > 1:  # 50 blocks a solve
        assert st["pc_launches"] == 2 * 50


PLAN_MEMORY = """
import resource, sys
sys.path.insert(0, sys.argv[1])
import cfdl
peak = lambda: resource.getrusage(resource.RUSAGE_SELF).ru_maxrss / 1024.0  # MiB
cfdl.UVWP.cavity(cfdl.Mesh.box(8).partition(2), mu=0.01).run(1, 1)
mesh = cfdl.Mesh.box(1, 1, 40000).partition(2)
before = peak()
eq = cfdl.UVWP.cavity(mesh, mu=0.01)
print("growth", peak() - before)
"""


def test_planning_memory_follows_the_batches():
    """A column of 40,000 cells is a chain of 10,000 tiles and as many steps;
    a table of every tile's every step is 1.2 GB a shape, the batches that
    exist are a few MB (64 MiB covers them and the context's own copies)."""
    out = subprocess.run([sys.executable, "-c", PLAN_MEMORY, os.path.dirname(cfdl.__path__[0])],
                         capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr[-2000:]
    growth = float(out.stdout.split("growth")[1])
    assert growth < 64.0, "%.0f MiB" % growth
