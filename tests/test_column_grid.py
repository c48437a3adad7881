"""The column kernels' grids, walked on the host (tests/cpp/column_grid.cpp):
every column exactly once, none outside, for whole and ragged widths, narrow
matrices alone and in groups, around every threshold of the rules."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def test_every_column_is_one_lanes(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("needs g++")
    exe = tmp_path / "column_grid"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", f"-I{ROOT / 'ascend-fft_amd' / 'csrc'}",
                    str(ROOT / "tests" / "cpp" / "column_grid.cpp"), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stdout
    assert int(run.stdout.split()[0]) > 100000
