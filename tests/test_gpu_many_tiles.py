"""Dense launches of more shared tiles than the workspace would hold a slot per tile and sharer for:
every workgroup of the launch has two partial-sum slots instead."""
import pytest

from tests.gpu_util import knobs
from tests.test_gpu_linear import _check_balanced

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,Kk,N,tile", [(2700, 256, 16640, 256), (1400, 384, 16640, 128)])
def test_more_tiles_than_slots_for_each(m, Kk, N, tile):
    if tile == 256:
        _check_balanced(m, Kk, N, True, tile)
    else:
        with knobs(BERTH_GEMM_ROWS256=0):
            _check_balanced(m, Kk, N, False, tile)
