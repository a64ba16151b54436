"""Device CSR construction at the edges of its tiles and digits: transposes
with empty and enormous rows, key widths from one bit a vertex up, rejected
pairs, kept memory reused across sizes, freed and shared by threads."""
import threading

import numpy as np
import pytest

from back40computing_amd import BfsError, CsrGraph
from back40computing_amd.primitives import DeviceCsr

pytestmark = pytest.mark.gpu


def same(d, g):
    h = d.to_host()
    assert np.array_equal(h.row_offsets, g.row_offsets)
    assert np.array_equal(h.column_indices, g.column_indices)


def host_transpose(nodes, src, dst):
    order = np.lexsort((src, dst))
    row = np.concatenate([[0], np.cumsum(np.bincount(dst, minlength=nodes))]).astype(np.int32)
    return CsrGraph.from_arrays(row, src[order].astype(np.int32))


@pytest.mark.parametrize("nodes,edges,where", [
    (1, 0, "all"), (1, 5, "all"), (2, 4095, "all"), (3, 4096, "all"), (300, 4097, "all"), (513, 12289, "all"),
    (50000, 9001, "one"), (50000, 20000, "last"), (200000, 5000, "sparse"), (1 << 20, 300000, "all"),
])
def test_transpose(gpu, nodes, edges, where):
    rng = np.random.default_rng(nodes + edges)
    src = {"all": rng.integers(0, nodes, edges), "one": np.full(edges, nodes // 3), "last": np.full(edges, nodes - 1),
           "sparse": (nodes // 7) * rng.integers(0, 7, edges)}[where].astype(np.int32)
    dst = rng.integers(0, nodes, edges).astype(np.int32)
    d = DeviceCsr.from_coo(nodes, src, dst)
    t = d.transpose()
    same(t, host_transpose(nodes, src, dst))
    same(t.transpose(), host_transpose(nodes, dst, src))


@pytest.mark.parametrize("nodes", [1, 2, 255, 512, 513, 1 << 17, (1 << 18) + 1])
def test_from_coo_key_widths(gpu, nodes):
    rng = np.random.default_rng(nodes)
    src, dst = (rng.integers(0, nodes, 30011).astype(np.int32) for _ in range(2))
    for sym, dedup, loops in ((False, False, False), (True, True, True), (True, False, True), (False, True, False)):
        d = DeviceCsr.from_coo(nodes, src, dst, symmetrize=sym, dedup=dedup, drop_self_loops=loops)
        same(d, CsrGraph.from_coo(nodes, src, dst, symmetrize=sym, dedup=dedup, drop_self_loops=loops))


def test_pairs_outside_are_rejected(gpu):
    src = np.zeros(5000, np.int32)
    for bad in (-1, 77, 2**31 - 1, -(2**31)):
        for at in (0, 4999):
            dst = np.ones(5000, np.int32)
            dst[at] = bad
            for a, b in ((src, dst), (dst, src)):
                with pytest.raises(BfsError):
                    DeviceCsr.from_coo(77, a, b, symmetrize=True)
    same(DeviceCsr.from_coo(77, src, np.ones(5000, np.int32)), CsrGraph.from_coo(77, src, np.ones(5000, np.int32)))


def test_kept_memory_over_sizes_and_threads(gpu):
    errors = []

    def work(seed):
        try:
            rng = np.random.default_rng(seed)
            for n in (100, 70000, 900, 250000, 1):
                src, dst = (rng.integers(0, 5000, n).astype(np.int32) for _ in range(2))
                d = DeviceCsr.from_coo(5000, src, dst, symmetrize=True, dedup=True)
                same(d, CsrGraph.from_coo(5000, src, dst, symmetrize=True, dedup=True))
                d.free()
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    work(0)
    threads = [threading.Thread(target=work, args=(s,)) for s in range(1, 5)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
