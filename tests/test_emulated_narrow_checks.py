"""Operands of the direct products and halves of the solves that do not fit each other (see run_narrow_checks.py), under the CPU emulation of the
kernels with AddressSanitizer."""
import subprocess
import sys

import pytest

from tests.emu import harness


@pytest.mark.parametrize("case", ["exponents", "few", "limbs", "halves", "refused"])
def test_operands(case):
    if harness.asan_runtime() is None:
        pytest.skip("no ASan runtime in this toolchain")
    harness.build()
    r = subprocess.run([sys.executable, "tests/emu/run_narrow_checks.py", case], env=harness.asan_env(), capture_output=True,
                       text=True, timeout=600, cwd=harness.HERE + "/../..")
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-6000:]
