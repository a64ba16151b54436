"""Batched top-down tiles: widths from one vertex to a whole workgroup, rows
around the grid tier's floor, and few tiles or few workgroups per counter
group, against the serial oracle."""
import numpy as np
import pytest

import oracle
from back40computing_amd import CsrGraph
from back40computing_amd.batch import Batch, GraphPool

pytestmark = pytest.mark.gpu


def fans(members, degree, seed):
    """0 -> members, each with `degree` edges to random targets, and back."""
    rng = np.random.default_rng(seed)
    targets = max(2, members * degree // 3)
    src = np.concatenate([np.zeros(members, np.int64), np.repeat(1 + np.arange(members), degree)])
    dst = np.concatenate([1 + np.arange(members), 1 + members + rng.integers(0, targets, members * degree)])
    return CsrGraph.from_coo(1 + members + targets, src, dst, symmetrize=True)


# rows of one, four and a workgroup's widths of edges, half a grid-tier chunk
# and one less, and a chunk and one more
GRAPHS = [(3000, 1, 1), (700, 4, 2), (257, 255, 3), (256, 257, 4), (9, 1023, 5), (9, 1025, 6), (5, 2049, 7), (1, 40000, 8)]


@pytest.mark.parametrize("mode", [Batch.PERSISTENT, Batch.GRAPH], ids=["persistent", "graph"])
@pytest.mark.parametrize("config", [{}, {"blocks_per_cu": 2, "grab_strided": 2, "tile_grab_max": 3},
                                    {"grid_gather_threshold": 64}, {"grid_gather_threshold": -1}],
                         ids=["default", "consecutive", "low", "never"])
def test_tile_widths(gpu, mode, config):
    graphs = [fans(*a) for a in GRAPHS]
    pool = GraphPool()
    for g in graphs:
        pool.add(g)
    b = Batch(pool, max_queries=40)
    if config:
        b.set_config(**config)
    for count in (1, 7, 40):
        gids = ((np.arange(count) * 5 + count) % len(graphs)).astype(np.int32)
        srcs = np.array([0 if q % 2 == 0 else graphs[g].nodes - 1 for q, g in enumerate(gids)], dtype=np.int32)
        for direction in (False, True):
            b.enact(gids, srcs, direction_optimizing=direction, mode=mode)
            for q, g in enumerate(gids):
                want = oracle.bfs(graphs[g].row_offsets, graphs[g].column_indices, int(srcs[q]))[0]
                assert oracle.compare(b.depths(q), want) == -1, (count, direction, q, GRAPHS[g])
    b.destroy()
    pool.destroy()
