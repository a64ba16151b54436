"""Adjacency levels of the LDS path (graphs of degree at most 8): record
widths of 4 and 8 words and one degree too many, frontiers that cross the
path's member limits, directed and self-looped graphs, small grids, against
the serial oracle."""
import numpy as np
import pytest

import back40computing_amd as b40c
from back40computing_amd import CsrGraph
from test_gpu_gather import check

pytestmark = pytest.mark.gpu


def regular(n, degree, seed):
    """Directed graph of out-degree `degree` everywhere (loops and duplicates among the edges)."""
    rng = np.random.default_rng(seed)
    return CsrGraph.from_coo(n, np.repeat(np.arange(n), degree), rng.integers(0, n, n * degree))


@pytest.mark.parametrize("degree", [1, 2, 4, 5, 8, 9])
def test_regular_graphs(gpu, degree):
    # frontiers grow past 1024 and 3072 members and shrink again
    check(regular(20011, degree, degree), sources=(0, 20010))


@pytest.mark.parametrize("width", [2, 33, 700])
def test_grid2d(gpu, width):
    check(CsrGraph.grid2d(width), sources=(0, width * width // 2))


def test_grid3d_frontiers_cross_the_limits(gpu):
    # levels of up to 1875 (between the limits) and 4800 members
    for width in (50, 80):
        check(CsrGraph.grid3d(width), sources=(0,))
    check(CsrGraph.grid3d(50), strategies=[b40c.EXPAND_CONTRACT, b40c.CONTRACT_EXPAND], fast_path_threshold=64)


def test_best_effort_and_bitmap_in_memory(gpu):
    g = CsrGraph.grid2d(120)
    check(g, cull_mode=b40c.CULL_BEST_EFFORT, sizing=64.0)
    check(g, fast_visited=2)
