"""Both tile sizes of the scan and copy-if kernels at the edges of their
ranges (one tile, the switch at 2^20 items, ragged ends, 4-byte offsets)
against torch-free closed forms and numpy."""
import numpy as np
import pytest

from back40computing_amd.primitives import SELECT_LESS, ScanEnactor
from hipmem import DeviceArray

pytestmark = pytest.mark.gpu

SWITCH = 1 << 20
SIZES = [1, 3, 4096, 4097, 16383, SWITCH - 1, SWITCH, SWITCH + 1, SWITCH + 8191, SWITCH + 16384, SWITCH + 16387]


@pytest.mark.parametrize("offset", [0, 1], ids=["aligned", "offset4"])
@pytest.mark.parametrize("n", SIZES)
def test_tile_edges(gpu, n, offset):
    e = ScanEnactor()
    x = np.random.default_rng(n).integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    incl = np.cumsum(x, dtype=np.uint32)
    d_in = DeviceArray(np.concatenate([np.zeros(offset, np.uint32), x]))
    d_out = DeviceArray(count=n + offset)
    src, dst = d_in.ptr.value + 4 * offset, d_out.ptr.value + 4 * offset
    for exclusive in (True, False):
        # twice: the second launch starts from the tile counter the first left
        for _ in range(2):
            assert e.scan(src, dst, n, exclusive) == int(incl[-1])
            assert np.array_equal(d_out.get()[offset:], incl - x if exclusive else incl)
    for comparand in (0, 1 << 30, 0xFFFFFFFF):
        kept = x[x < np.uint32(comparand)]
        assert e.copy_if(src, dst, n, SELECT_LESS, comparand) == len(kept)
        assert np.array_equal(d_out.get()[offset:offset + len(kept)], kept)
    e.destroy()
