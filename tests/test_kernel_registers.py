"""Vector registers of the built transform kernels.

A SIMD has 512 a lane: up to 96 registers leave it five waves, up to 128 four.
The plain FFT's kernels for lengths of the factors 2, 3 and 5 (and of primes
above 13) do without the butterflies of 7, 11 and 13, which take 16 to 32
registers more.
"""

import re
import shutil
import subprocess
from pathlib import Path

import pytest

from bldfm_amd import build

TOOLS = {n: shutil.which(n) or f"/opt/rocm/llvm/bin/{n}" for n in ("llvm-objdump", "llvm-readelf")}


@pytest.fixture(scope="module")
def registers(tmp_path_factory):
    """{mangled kernel name: registers} of the library's gfx950 code."""
    if not all(Path(t).exists() for t in TOOLS.values()):
        pytest.skip("no LLVM binary tools")
    if not build.LIB.exists():
        build.build()
    d = tmp_path_factory.mktemp("code")
    shutil.copy(build.LIB, d / "lib.so")
    subprocess.run([TOOLS["llvm-objdump"], "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    regs = {}
    for f in d.glob("lib.so.*gfx950*"):
        notes = subprocess.run([TOOLS["llvm-readelf"], "--notes", str(f)], check=True, capture_output=True, text=True).stdout
        for kernel in re.split(r"\n\s+- \.agpr_count", notes)[1:]:
            name = re.search(r"\n\s+\.name:\s+(\S+)", kernel).group(1)
            regs[name] = int(re.search(r"\n\s+\.vgpr_count:\s+(\d+)", kernel).group(1))
    return regs


@pytest.mark.parametrize("element", ["HIP_vector_typeIdLj2E", "HIP_vector_typeIfLj2E"])
@pytest.mark.parametrize("kernel,most", [
    ("11k_fft2_rowsILi8ELi256E", 100), ("11k_fft2_colsILi8ELi256E", 96), ("11k_fft2_colsILi10ELi1024E", 96),
    ("16k_fft2_col_tilesILi4E", 96), ("16k_fft2_col_tilesILi8E", 96)])
def test_plain_fft_of_smooth_lengths_pays_for_no_prime_butterfly(registers, kernel, element, most):
    found = {n: r for n, r in registers.items() if re.search(kernel + "(Lb[01]E)?15" + element, n)}
    assert found
    assert min(found.values()) <= most, found
