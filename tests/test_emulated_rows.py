"""Products of one or two rows in large batches (a wave per column or slice) under the CPU emulation of the kernels
(AddressSanitizer), against the oracle: one and two words per lane, one slice and several."""
import subprocess
import sys

import pytest

from tests.emu import harness


@pytest.mark.parametrize("case", ["few 8 2560 1 1 2", "few 24 1024 1 1 2", "few 33 512 1 2 3", "few 49 256 1 1 3",
                                  "few 49 128 1 1 129"])
def test_rows(case):
    if harness.asan_runtime() is None:
        pytest.skip("no ASan runtime in this toolchain")
    harness.build()
    r = subprocess.run([sys.executable, "tests/emu/run_rows.py", *case.split()], env=harness.asan_env(), capture_output=True,
                       text=True, timeout=600, cwd=harness.HERE + "/../..")
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-6000:]
