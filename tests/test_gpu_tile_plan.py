"""The tile shape and layer-aligned cuts the sweep schedules are planned with,
against the oracle bit for bit: uneven and one-layer boxes, distorted cells,
more layers than a tile holds, edges one past a tile's, a mesh whose layers
are no planes (three blocks around an edge)."""
import pytest

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
