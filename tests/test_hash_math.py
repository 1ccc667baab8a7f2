"""The parts of the device hash that a host can evaluate too (strata-concurrent_amd/csrc/sc_hash_math.hpp), compiled from
the kernels' own header into tests/cpp/bin/hash_math_test and compared with plain loops there."""
import subprocess
from pathlib import Path

import pytest

PROGRAM = Path(__file__).resolve().parent / "cpp" / "bin" / "hash_math_test"


@pytest.mark.parametrize("name", ["extents"])
def test_hash_math(name):
    run = subprocess.run([str(PROGRAM), name], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0, run.stdout + run.stderr
