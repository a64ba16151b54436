"""Searches of small graphs run on fewer workgroups; what the caller sees of
the grid stays that of the full one."""
import numpy as np
import pytest

import back40computing_amd as b40c
import oracle
from back40computing_amd import CsrGraph, CsrProblem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [140, 300, 600, 720])
def test_hybrid_stays_persistent_below_the_full_grids_threshold(gpu, n):
    # a complete graph: one level's edges are nearly all, fewer than 4 items per thread of 256 workgroups
    a = np.repeat(np.arange(n), n - 1)
    b = (a + 1 + np.tile(np.arange(n - 1), n)) % n
    g = CsrGraph.from_coo(n, a, b)
    p = CsrProblem().from_host_problem(g)
    p.reset(b40c.EDGE_FRONTIERS, 1.3)
    st = p.enact(b40c.HYBRID, 3)
    assert oracle.compare(p.extract_depths(), oracle.bfs(g.row_offsets, g.column_indices, 3)[0]) == -1
    # contract-expand alone: one launch, the source and every edge queued once
    assert st.kernel_launches == 1
    assert st.total_queued == 1 + g.edges
