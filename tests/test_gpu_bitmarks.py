"""Bit marks (large steps of graphs whose visited bitmap fits LDS): graphs at
the edges of their rule and of the bitmap's words, hubs beside short rows,
every strategy fused and per level, against the serial oracle."""
import numpy as np
import pytest

import back40computing_amd as b40c
from back40computing_amd import CsrGraph, _native
from test_gpu_gather import check

pytestmark = pytest.mark.gpu


def layered(members, targets, edges, hubs, isolated=0):
    """0 -> members -> `edges` random edges to targets (the first `hubs`
    members hold half of them), then one more level back to a few vertices."""
    rng = np.random.default_rng(edges + members)
    n = 1 + members + targets + isolated
    per = np.where(np.arange(edges) < edges // 2, rng.integers(0, max(hubs, 1), edges),
                   rng.integers(0, members, edges))
    src = np.concatenate([np.zeros(members, np.int64), 1 + per, 1 + members + np.arange(targets)])
    dst = np.concatenate([1 + np.arange(members), 1 + members + rng.integers(0, targets, edges),
                          1 + rng.integers(0, members, targets)])
    return CsrGraph.from_coo(n, src, dst)


@pytest.mark.parametrize("members,targets,edges,hubs,isolated", [
    (1500, 60001, (1 << 20) + 5, 3, 0),        # the smallest marked step, a few long rows
    (40000, 65537, 1 << 21, 40000, 3),         # rows of tens of edges
    (1200000 // 4, 500000, 1300000, 100, 17),  # most rows shorter than a lane group
    (700, 31, (1 << 20) + 100000, 700, 0),     # few targets, all duplicates
])
def test_layered(gpu, members, targets, edges, hubs, isolated):
    g = layered(members, targets, edges, hubs, isolated)
    check(g)
    check(g, pred=False, strategies=[b40c.EXPAND_CONTRACT, b40c.TWO_PHASE], cull_mode=b40c.CULL_BEST_EFFORT,
          sizing=4.0)


@pytest.mark.parametrize("nodes", [_native.FAST_VISITED_MAX, _native.FAST_VISITED_MAX + 1])
def test_largest_bitmap(gpu, nodes):
    rng = np.random.default_rng(nodes)
    m = 4 * nodes
    g = CsrGraph.from_coo(nodes, rng.integers(0, nodes, m), rng.integers(0, nodes, m), symmetrize=True)
    check(g, strategies=[b40c.EXPAND_CONTRACT, b40c.CONTRACT_EXPAND, b40c.TWO_PHASE], sources=(1,))


def test_rmat_repeated(gpu):
    # marks, slabs and counters left by one search do not show in the next
    g = CsrGraph.rmat(17, 24, seed=9)
    check(g, sources=tuple(int(s) for s in g.sample_sources(3, seed=2)))


@pytest.mark.parametrize("targets", [20000, (1 << 18) - 1501, (1 << 18) - 1500])
@pytest.mark.parametrize("below", [0, 1])
def test_smallest_marked_step(gpu, targets, below):
    # the second step has exactly the edges of the rule, or one less
    work = (1 << 16) + (1501 + targets) // 2 - below
    check(layered(1500, targets, work, 40))
