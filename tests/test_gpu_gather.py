"""Grid-wide steps at the edges of their forms: tiles of one row, a full tile
and one row more, rows around the grid tier's thresholds, rows heavy enough
for a tile to publish, and long chains of light steps; every persistent
strategy and the launches per step against the serial oracle."""
import numpy as np
import pytest

import back40computing_amd as b40c
import oracle
from back40computing_amd import CsrGraph, CsrProblem, _native

pytestmark = pytest.mark.gpu

STRATEGIES = [b40c.EXPAND_CONTRACT, b40c.CONTRACT_EXPAND, b40c.TWO_PHASE, b40c.HYBRID, b40c.DIRECTION_OPTIMIZING]


def check(g, pred=True, strategies=STRATEGIES, sources=(0,), sizing=1.3, **cfg):
    row, col = g.row_offsets, g.column_indices
    for strategy in strategies:
        p = CsrProblem(mark_predecessors=pred).from_host_problem(g)
        if cfg:
            p.set_config(**cfg)
        p.reset(_native.load().bfs_strategy_frontier_type(strategy), sizing)
        for src in sources:
            expect, levels, _ = oracle.bfs(row, col, src)
            for fused in (True, False):
                st = p.enact(strategy, src, fused=fused)
                assert oracle.compare(p.extract_depths(), expect) == -1, (strategy, fused, src)
                assert st.search_depth == levels, (strategy, fused, src)
                if pred:
                    assert oracle.check_preds(row, col, expect, p.extract_results()) == -1, (strategy, fused, src)
        p.destroy()


def fan(members, degrees, tail):
    """0 -> members vertices -> degrees[i] targets each (drawn from `tail` vertices)."""
    rng = np.random.default_rng(members)
    first, last = 1, 1 + members
    src = [np.zeros(members, np.int64)]
    dst = [np.arange(first, last)]
    deg = np.resize(np.asarray(degrees), members)
    src.append(np.repeat(np.arange(first, last), deg))
    dst.append(last + rng.integers(0, tail, int(deg.sum())))
    return CsrGraph.from_coo(last + tail, np.concatenate(src), np.concatenate(dst))


@pytest.mark.parametrize("members,degrees,tail", [
    (1025, [1], 64),                       # just past the LDS path, one edge a row
    (1040, [0, 0, 3], 5000),               # empty rows between
    (4113, [17], 40000),                   # a few rows per workgroup
    (1500, [2, 2047, 2, 2048, 2049], 90000),   # around the grid tier of narrow steps
    (2000, [1] * 1999 + [70000], 80000),   # one hub among single edges
    (9000, [60, 511, 512, 513], 200000),   # tiles heavy enough to publish rows of 512
    (131072 + 17, [2, 1], 50000),          # one tile per workgroup and a few more
])
def test_fan_levels(gpu, members, degrees, tail):
    check(fan(members, degrees, tail))


def test_wide_items(gpu):
    # edge frontiers past one 2048-item tile per workgroup, with duplicates
    check(fan(3000, [200], 1500), strategies=[b40c.CONTRACT_EXPAND, b40c.TWO_PHASE, b40c.HYBRID])


def test_long_chain_of_light_steps(gpu):
    # 40 levels of 3000 vertices, two forward edges and one back edge each
    rng = np.random.default_rng(4)
    w, d = 3000, 40
    v = np.arange(w * (d - 1)).reshape(d - 1, w)
    nxt = (np.arange(1, d)[:, None] * w + rng.integers(0, w, (d - 1, 2 * w))).ravel()
    src = np.concatenate([np.zeros(w - 1, np.int64), np.tile(v, (1, 2)).ravel(), nxt])
    dst = np.concatenate([np.arange(1, w), nxt, np.tile(v, (1, 2)).ravel()])
    g = CsrGraph.from_coo(w * d, src, dst)
    check(g, sources=(0, 7))
    check(g, pred=False, strategies=[b40c.EXPAND_CONTRACT, b40c.DIRECTION_OPTIMIZING], cull_mode=b40c.CULL_BEST_EFFORT,
          sizing=16.0)


def test_search_depth_of_sinks(gpu):
    # the deepest vertices have no neighbours at all
    src = np.concatenate([np.zeros(3000, np.int64), np.repeat(np.arange(1, 3001), 2)])
    dst = np.concatenate([np.arange(1, 3001), 3001 + np.arange(6000)])
    check(CsrGraph.from_coo(9001, src, dst))
