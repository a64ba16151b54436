"""Transposes of graphs with far fewer edges than vertices, or long runs of
empty rows: tiles on both sides of the rows an edge that a tile walks, and
their device time beside that of building the same pairs."""
import numpy as np
import pytest

from back40computing_amd.primitives import DeviceCsr
from test_gpu_csr_forms import host_transpose, same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nodes,edges", [(1 << 21, 1000), (20000000, 5000), (1 << 21, 4097), (5 * 16384, 4096),
                                         (5 * 16384 + 700, 9000), (1 << 20, 200000)])
@pytest.mark.parametrize("where", ["all", "ends"])
def test_transpose_of_mostly_empty_rows(gpu, nodes, edges, where):
    # tiles on both sides of the rows an edge that are walked; long runs of empty rows inside a tile
    rng = np.random.default_rng(nodes + edges)
    src = rng.integers(0, nodes, edges)
    if where == "ends":
        src = np.where(src % 2 == 0, src % 50, nodes - 1 - src % 50)
    src, dst = src.astype(np.int32), rng.integers(0, nodes, edges).astype(np.int32)
    d = DeviceCsr.from_coo(nodes, src, dst)
    same(d.transpose(), host_transpose(nodes, src, dst))


@pytest.mark.parametrize("nodes,edges", [(1 << 21, 1000), (20000000, 5000)])
def test_sparse_transpose_costs_no_more_than_its_build(gpu, nodes, edges):
    # fewer sorting passes than the build of the same pairs, and no copy of them
    rng = np.random.default_rng(edges)
    src, dst = (rng.integers(0, nodes, edges).astype(np.int32) for _ in range(2))
    built, transposed = [], []
    for _ in range(5):
        d = DeviceCsr.from_coo(nodes, src, dst)
        built.append(d.build_ms)
        transposed.append(d.transpose().build_ms)
    assert min(transposed) <= 2 * min(built), (transposed, built)
