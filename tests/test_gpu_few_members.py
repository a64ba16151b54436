"""Levels of few vertices launched step by step: rows around a wave's length,
members around a workgroup's, against the serial oracle."""
import pytest

from test_gpu_gather import check, fan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("members", [1, 15, 17, 511, 512, 513])
@pytest.mark.parametrize("degrees", [[63, 64, 65], [1, 2047, 300, 0], [64]])
def test_few_members(gpu, members, degrees):
    check(fan(members, degrees, 3000))
    check(fan(members, degrees, 100), pred=False, grid_gather_threshold=-1)
