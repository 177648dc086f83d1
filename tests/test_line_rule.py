"""The rule that runs a pass's lines as chirps, against measured passes."""

import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_chirps_are_taken_where_they_measured_faster(tmp_path):
    exe = tmp_path / "line_chirp_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-o", str(exe),
                    str(ROOT / "tests" / "native" / "line_chirp_check.cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
