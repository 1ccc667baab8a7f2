"""The parts of the device hash that a host can evaluate too (strata-concurrent_amd/csrc/sc_hash_math.hpp: a level's maps, the
weights and powers of the sums, the search of a workgroup's extent), compiled from the kernels' own header into
tests/cpp/bin/hash_math_test and compared with the byte loop and plain searches there."""
import subprocess
from pathlib import Path

import pytest

PROGRAM = Path(__file__).resolve().parent / "cpp" / "bin" / "hash_math_test"


@pytest.mark.parametrize("name", ["levels", "sums", "powers", "extents"])
def test_hash_math(name):
    run = subprocess.run([str(PROGRAM), name], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0, run.stdout + run.stderr
