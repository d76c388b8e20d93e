"""The routes of small calls against the general ones under the CPU emulation of the kernels (AddressSanitizer)."""
import subprocess
import sys

import pytest

from tests.emu import harness


@pytest.mark.parametrize("case", ["fused", "native", "blocks", "tile"])
def test_route(case):
    if harness.asan_runtime() is None:
        pytest.skip("no ASan runtime in this toolchain")
    harness.build()
    r = subprocess.run([sys.executable, "tests/emu/run_routes.py", case], env=harness.asan_env(), capture_output=True,
                       text=True, timeout=300, cwd=harness.HERE + "/../..")
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-6000:]
