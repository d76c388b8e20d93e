"""sdpv_exact_dot under the CPU emulation of the kernels (AddressSanitizer), against Python integers."""
import subprocess
import sys

import pytest

from tests.emu import harness


@pytest.mark.parametrize("case", ["exact_dot 2 1 34 2 5 128 3", "exact_dot 25 1 2 1 40 52 1", "exact_dot 63 1 2 1 3 128 1",
                                  "exact_dot 49 256 1 1 2 100 1", "exact_dot 3 1 2 1 0 8 1"])
def test_exact_dot(case):
    if harness.asan_runtime() is None:
        pytest.skip("no ASan runtime in this toolchain")
    harness.build()
    r = subprocess.run([sys.executable, "tests/emu/run_rows.py", *case.split()], env=harness.asan_env(), capture_output=True,
                       text=True, timeout=600, cwd=harness.HERE + "/../..")
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-6000:]
