"""Threads of the tile kernels: the documented settings take effect (and change no result), and a tile that fits in LDS
beside the operands of fewer waves is factored there by fewer waves. Run under the CPU emulation of the kernels,
against the oracle."""
import subprocess
import sys

import pytest

from tests.emu import harness


@pytest.mark.parametrize("L,BT,settings,launches", [
    (2, 9, {}, "1 1"),                                           # inverse 512, factorisation 1024 threads
    (2, 9, dict(SDPV_TILE_THREADS="256", SDPV_INV_THREADS="1024"), "0 1"),
    (2, 9, dict(SDPV_TILE_THREADS="512", SDPV_INV_THREADS="256"), "1 0"),
    (2, 9, dict(SDPV_TILE_LANE_PAIRS="20"), "1 1"),
    (2, 51, {}, "2 0"),                                          # 1024 threads' operands do not fit beside the tile
])
def test_tile_launches(L, BT, settings, launches):
    if harness.asan_runtime() is None:
        pytest.skip("no ASan runtime in this toolchain")
    harness.build()
    r = subprocess.run([sys.executable, "tests/emu/run_tile_launch.py", str(L), str(BT)], env={**harness.asan_env(), **settings},
                       capture_output=True, text=True, timeout=600, cwd=harness.HERE + "/../..")
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-6000:]
    assert r.stdout.splitlines()[-1] == launches
