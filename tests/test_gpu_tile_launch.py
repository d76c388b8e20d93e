"""Tiles that fit in LDS beside the operands of eight or four waves, not of sixteen, against the oracle, bit for bit."""
import pytest

from tests.intutil import spd_tile
from tests.test_gpu_tile import tile_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,BT", [(2, 52), (8, 47), (14, 43), (24, 38), (36, 34)])
def test_larger_tiles_on_fewer_waves(L, BT):
    tile_parity([spd_tile(BT, 12, L, 32 * L - 40)], L, BT)
