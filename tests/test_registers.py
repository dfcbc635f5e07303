"""Registers of built kernels whose speed hangs on how many of their waves a SIMD holds (read from the built library)."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from lab import hip

LLVM = Path("/opt/rocm/llvm/bin")


@pytest.fixture(scope="module")
def vgprs(tmp_path_factory):
    """Kernel symbol -> VGPRs, from the library's gfx950 code object."""
    d = tmp_path_factory.mktemp("code")
    shutil.copy(hip.LIB_PATH, d / "lib.so")
    subprocess.run([LLVM / "llvm-objdump", "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    (code,) = d.glob("*gfx950*")
    notes = subprocess.run([LLVM / "llvm-readelf", "--notes", code], check=True, capture_output=True, text=True).stdout
    return {re.search(r"\.name:\s+(\S+)", k)[1]: int(re.search(r"\.vgpr_count:\s+(\d+)", k)[1])
            for k in notes.split("- .agpr_count")[1:]}


def test_o_product_merge_holds_three_waves_per_simd(vgprs):
    """The O products with the attention merge in their prologue (k_gemv, prologue 2, epilogue 6): 195 VGPRs (two waves)
    cost 6 to 14 % at short contexts."""
    n = [v for k, v in vgprs.items() if re.search(r"k_gemvILi\dELi\dELi\dELi\dELi2ELi6E", k)]
    assert len(n) == 8 and max(n) <= 512 // 3 // 8 * 8
