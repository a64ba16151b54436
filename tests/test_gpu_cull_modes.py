"""Best-effort culls outside chained compaction claim as exact ones do: the
same labels, the same number of queued items, in queues of the same size."""
import pytest

import back40computing_amd as b40c
import oracle
from back40computing_amd import CsrGraph, CsrProblem, _native
from test_gpu_gather import STRATEGIES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("strategy", STRATEGIES)
@pytest.mark.parametrize("compaction", [1, 2])
def test_best_effort_queues_what_exact_does(gpu, strategy, compaction):
    if compaction == 2 and strategy in (b40c.TWO_PHASE, b40c.HYBRID):
        pytest.skip("chained contractions let duplicates through")
    for g in (CsrGraph.rmat(17, 24, seed=4), CsrGraph.grid2d(200), CsrGraph.random(30001, 200003, seed=5)):
        src = int(g.sample_sources(1, seed=3)[0])
        expect, _, _ = oracle.bfs(g.row_offsets, g.column_indices, src)
        p = CsrProblem(mark_predecessors=True).from_host_problem(g)
        p.reset(_native.load().bfs_strategy_frontier_type(strategy), 1.3)
        for fused in (True, False):
            queued = []
            for cull in (b40c.CULL_EXACT, b40c.CULL_BEST_EFFORT):
                p.set_config(cull_mode=cull, compaction=compaction)
                queued.append(p.enact(strategy, src, fused=fused).total_queued)
                assert oracle.compare(p.extract_depths(), expect) == -1
                assert oracle.check_preds(g.row_offsets, g.column_indices, expect, p.extract_results()) == -1
            assert queued[0] == queued[1], (fused, queued)
        p.destroy()
