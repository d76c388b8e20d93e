"""Sums of products with one or two columns over segments, kept as exact words (one and two per lane), under the CPU
emulation of the kernels (AddressSanitizer), against the oracle."""
import subprocess
import sys

import pytest

from tests.emu import harness


@pytest.mark.parametrize("case", ["ksum 3 5 2", "ksum 26 4 1", "ksum 33 3 2", "ksum 63 3 1"])
def test_ksum(case):
    if harness.asan_runtime() is None:
        pytest.skip("no ASan runtime in this toolchain")
    harness.build()
    r = subprocess.run([sys.executable, "tests/emu/run_rows.py", *case.split()], env=harness.asan_env(), capture_output=True,
                       text=True, timeout=600, cwd=harness.HERE + "/../..")
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-6000:]
