"""The arithmetic of the search kernels' staged boxes on the host, through its C++
test program tests/cpp/cell_test."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BIN = os.path.join(ROOT, "tests", "cpp", "cell_test")


@pytest.mark.parametrize("suite", ["Cells", "Keys"])
def test_stage_cells(suite):
    if not os.path.exists(BIN):
        subprocess.run(["make", "-s", "-C", os.path.dirname(BIN), BIN], check=True)
    p = subprocess.run([BIN, suite], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout + p.stderr
