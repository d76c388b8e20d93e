"""Tiles that fit in LDS beside the operands of eight or four waves, not of sixteen, and the settings of the tile
kernels' threads, against the oracle, bit for bit."""
import os
import subprocess
import sys

import pytest

from tests.intutil import spd_tile
from tests.test_gpu_tile import tile_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,BT", [(2, 52), (8, 47), (14, 43), (24, 38), (36, 34)])
def test_larger_tiles_on_fewer_waves(L, BT):
    tile_parity([spd_tile(BT, 12, L, 32 * L - 40)], L, BT)


@pytest.mark.parametrize("settings", [dict(SDPV_TILE_THREADS="256", SDPV_INV_THREADS="1024", SDPV_TILE_LANE_PAIRS="200"),
                                      dict(SDPV_TILE_THREADS="512", SDPV_INV_THREADS="256", SDPV_TILE_LANE_PAIRS="9")])
def test_settings_change_no_result(settings):
    code = ("from tests.intutil import spd_tile; from tests.test_gpu_tile import tile_parity\n"
            "for L, BT in ((24, 32), (40, 30), (9, 45)):\n"
            "    tile_parity([spd_tile(BT, 12, L + b, 32 * L - 40) for b in range(2)], L, BT)\n")
    r = subprocess.run([sys.executable, "-c", code], env={**os.environ, **settings}, capture_output=True, text=True, timeout=100,
                       cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    assert r.returncode == 0, r.stderr[-3000:]
