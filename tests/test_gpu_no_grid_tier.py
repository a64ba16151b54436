"""Searches with the grid tier off (grid_gather_threshold -1): the steps that
share long rows all the same (few vertices, bit marks) and those that do not."""
import numpy as np
import pytest

from back40computing_amd import CsrGraph
from back40computing_amd.batch import Batch, GraphPool
import oracle
from test_gpu_bitmarks import layered
from test_gpu_gather import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("members,targets,edges,hubs", [
    (1500, 60001, (1 << 20) + 5, 3),        # bit marks, rows of 100 k edges
    (300, 60001, 50000, 3),                 # few vertices
    (200000, 30001, 90000, 2),              # many vertices, below the bit marks' rule
])
def test_no_grid_tier(gpu, members, targets, edges, hubs):
    check(layered(members, targets, edges, hubs), pred=False, grid_gather_threshold=-1)


def test_batch_rows_around_its_thresholds(gpu):
    # one vertex leads to tiles of more than 32768 edges with rows of 512 to 1023 among short ones
    rng = np.random.default_rng(7)
    deg = np.concatenate([rng.integers(500, 1100, 120), np.ones(3000, np.int64)])
    src = np.concatenate([np.zeros(len(deg), np.int64), np.repeat(1 + np.arange(len(deg)), deg)])
    dst = np.concatenate([1 + np.arange(len(deg)), 1 + len(deg) + rng.integers(0, 50000, int(deg.sum()))])
    g = CsrGraph.from_coo(1 + len(deg) + 50000, src, dst)
    expect = [oracle.bfs(g.row_offsets, g.column_indices, s)[0] for s in (0, 1, 121)]
    pool = GraphPool()
    pool.add(g)
    b = Batch(pool, max_queries=3)
    for t in (-1, 1, 256, 2048):
        b.set_config(grid_gather_threshold=t)
        b.enact(np.zeros(3, np.int32), np.array([0, 1, 121], np.int32), direction_optimizing=False)
        for q in range(3):
            assert oracle.compare(b.depths(q), expect[q]) == -1, (t, q)
