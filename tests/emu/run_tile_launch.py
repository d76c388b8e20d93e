"""One emulated tile factorisation and inverse against the oracle, and the launches with 512 and 1024 threads that it
took. Usage: run_tile_launch.py L BT"""
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__)))))
from tests.emu import harness  # noqa: E402

lib = harness.install()
import torch  # noqa: E402

import tests.test_gpu_tile as T  # noqa: E402
from tests.intutil import spd_tile  # noqa: E402

if __name__ == "__main__":
    L, BT = int(sys.argv[1]), int(sys.argv[2])
    T.cu = torch.from_numpy
    T.tile_parity([spd_tile(BT, 6, L, 32 * L - 40)], L, BT)
    print(lib.emu_launched(512), lib.emu_launched(1024))
