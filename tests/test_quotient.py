"""The kernels' division by a shared divisor (``corrected_quotient``, economize_amd/csrc/fp8_codec.hpp) against IEEE
division on the CPU, where they use it in its place."""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_corrected_quotients_equal_ieee_division(tmp_path: Path) -> None:
    exe = tmp_path / "quotient"
    has = Path("/proc/cpuinfo").read_text().split()
    vector = [flag for name, flag in (("fma", "-mfma"), ("avx2", "-mavx2")) if name in has]
    subprocess.run(["g++", "-O3", "-std=c++17", "-fopenmp", *vector, "-ffp-contract=off",
                    str(ROOT / "tests/native/quotient_check.cpp"), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split() == ["0"]
