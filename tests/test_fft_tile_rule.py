"""The plain 2-D FFT's rule for columns per workgroup."""

import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_column_tiles_are_not_mostly_empty(tmp_path):
    exe = tmp_path / "fft2_tile_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-o", str(exe),
                    str(ROOT / "tests" / "native" / "fft2_tile_check.cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
