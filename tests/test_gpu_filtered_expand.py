"""Two-phase levels whose expand step filters as well, against the form that
keeps a filter step (chained compaction): the same depths, the same count of
queued elements, and the same refusal of an edge queue that cannot hold a
level's unfiltered edges."""
import numpy as np
import pytest

import oracle
import back40computing_amd as b40c
from back40computing_amd import CsrGraph, CsrProblem

pytestmark = pytest.mark.gpu


def clique(n):
    i, j = np.divmod(np.arange(n * n), n)
    return CsrGraph.from_coo(n, i[i != j], j[i != j])


def star_of_hubs():
    # a hub of three grid-tier chunks and one more edge, and rows around the
    # length from which a narrow step's tiles share them
    src = np.concatenate([np.zeros(6145, np.int64), np.repeat([1, 2, 3], [255, 256, 257])])
    dst = np.concatenate([1 + np.arange(6145), 6146 + np.arange(255), 6200 + np.arange(256), 6100 + np.arange(257)])
    return CsrGraph.from_coo(6500, src, dst, symmetrize=True)


@pytest.mark.parametrize("make", [lambda: clique(150), star_of_hubs, lambda: CsrGraph.rmat(14, 16, seed=3),
                                  lambda: CsrGraph.random(70001, 300000, seed=4), lambda: CsrGraph.grid3d(31)],
                         ids=["clique", "hubs", "rmat", "random", "grid3d"])
@pytest.mark.parametrize("pred", [False, True], ids=["depth", "pred"])
@pytest.mark.parametrize("strategy,fused", [(b40c.TWO_PHASE, True), (b40c.TWO_PHASE, False), (b40c.HYBRID, True)],
                         ids=["fused", "iter", "hybrid"])
def test_counts_and_depths(gpu, make, pred, strategy, fused):
    g = make()
    want = oracle.bfs(g.row_offsets, g.column_indices, 0)[0]
    queued = []
    for compaction in (1, 2):
        p = CsrProblem(mark_predecessors=pred).from_host_problem(g)
        p.set_config(compaction=compaction, saturation_threshold=300)
        p.reset(b40c.EDGE_FRONTIERS, 1.3)
        queued.append(p.enact(strategy, 0, fused=fused).total_queued)
        assert oracle.compare(p.extract_depths(), want) == -1
        p.destroy()
    assert queued[0] == queued[1]


@pytest.mark.parametrize("compaction", [1, 2])
@pytest.mark.parametrize("strategy,fused", [(b40c.TWO_PHASE, True), (b40c.TWO_PHASE, False)], ids=["fused", "iter"])
def test_edges_past_the_queue(gpu, compaction, strategy, fused):
    # nearly every edge of the second level leads back: few pass the filter,
    # none of them past the queue's end
    g = clique(150)
    p = CsrProblem().from_host_problem(g)
    p.set_config(compaction=compaction)
    p.reset(b40c.EDGE_FRONTIERS, 0.5)
    with pytest.raises(b40c.BfsError, match="overflow"):
        p.enact(strategy, 0, fused=fused)
    p.reset(b40c.EDGE_FRONTIERS, 1.0)
    p.enact(strategy, 0, fused=fused)
    assert oracle.compare(p.extract_depths(), oracle.bfs(g.row_offsets, g.column_indices, 0)[0]) == -1
    p.destroy()


@pytest.mark.parametrize("members", [2047, 2048, 2049, 131072, 131073])
@pytest.mark.parametrize("cull", [b40c.CULL_EXACT, b40c.CULL_BEST_EFFORT], ids=["exact", "best_effort"])
def test_rows_of_a_step_by_waves(gpu, members, cull):
    # 0 -> members, whose rows have 0, 1, 31, 32, 33 and 511 to 513 edges: as
    # many members as the waves of a full grid, and a full run for each wave
    rng = np.random.default_rng(members)
    deg = rng.integers(0, 3, members)
    deg[rng.choice(members, 40, replace=False)] = np.tile([31, 32, 33, 511, 512, 513, 64, 2049], 5)
    targets = 600000
    src = np.concatenate([np.zeros(members, np.int64), np.repeat(1 + np.arange(members), deg)])
    dst = np.concatenate([1 + np.arange(members), 1 + members + rng.integers(0, targets, int(deg.sum()))])
    g = CsrGraph.from_coo(1 + members + targets, src, dst)
    p = CsrProblem(mark_predecessors=members % 2 == 0).from_host_problem(g)
    p.set_config(cull_mode=cull)
    p.reset(b40c.EDGE_FRONTIERS, 2.0)
    p.enact(b40c.TWO_PHASE, 0)
    assert oracle.compare(p.extract_depths(), oracle.bfs(g.row_offsets, g.column_indices, 0)[0]) == -1
    p.destroy()
