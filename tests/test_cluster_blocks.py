"""Even split of structured blocks into element clusters
(weldformfem_amd/csrc/wfx_cluster.cpp), on the CPU: blocks whose edges are
no multiples of the standing 16 x 4 x 4 brick, thin and long ones, blocks next
to others, and a block with a cell missing (no block any more).  Every plan
passes the same checks as the others, and where a block is split evenly its
clusters are whole bricks.
"""
import numpy as np
import pytest

from test_cluster_plan import check_plan, plan, planner  # noqa: F401
from weldformfem_amd import workloads

BLOCKS = [(21, 17, 13), (26, 22, 18), (43, 19, 9), (37, 11, 7), (1, 1, 700), (3, 200, 1), (257, 1, 1), (19, 23, 2), (16, 16, 1)]


def bricks(p, el, size):
    """each cluster's cells: None unless they are a box"""
    ijk = np.stack(np.unravel_index(np.arange(len(el)), size[::-1]), axis=1)[:, ::-1]
    for c in range(len(p["eoff"]) - 1):
        b = ijk[p["s2o"][p["eoff"][c]:p["eoff"][c + 1]]]
        yield (b.max(axis=0) - b.min(axis=0) + 1).prod() == len(b)


@pytest.mark.parametrize("size", BLOCKS)
def test_block(planner, tmp_path, size):
    x, el = workloads.hexa_box(*size, 0.05)
    p = plan(planner, tmp_path, x, el, 8)
    check_plan(p, el, len(x), 8)
    whole = list(bricks(p, el, size))
    if size in BLOCKS[:3]:
        assert all(whole)
        # and that is fewer slots and clusters than the runs of 256 along bricks of 16 x 4 x 4
        cells = [np.ceil(s / b) for s, b in zip(size, (16, 4, 4))]
        assert len(whole) <= np.prod(cells)


def test_block_with_a_missing_cell(planner, tmp_path):
    x, el = workloads.hexa_box(21, 17, 13, 0.05)
    el = np.delete(el, 1234, axis=0)
    p = plan(planner, tmp_path, x, el, 8)
    check_plan(p, el, len(x), 8)


def test_small_clusters(planner, tmp_path):
    x, el = workloads.hexa_box(9, 7, 5, 0.05)
    check_plan(plan(planner, tmp_path, x, el, 8, cs=7), el, len(x), 8, cs=7)


def test_blocks_side_by_side(planner, tmp_path):
    xa, ea = workloads.hexa_box(21, 17, 13, 0.05)
    xb, eb = workloads.hexa_box(11, 9, 23, 0.05, (3.0, 0.0, 0.0))
    el = np.concatenate([ea, eb + len(xa)])
    both = plan(planner, tmp_path, np.concatenate([xa, xb]), el, 8)
    check_plan(both, el, len(xa) + len(xb), 8)
    alone = plan(planner, tmp_path, xb, eb, 8)
    np.testing.assert_array_equal(both["s2o"][len(ea):] - len(ea), alone["s2o"])
    np.testing.assert_array_equal(both["lslot"][len(ea) * 8:], alone["lslot"])
