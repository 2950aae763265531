"""The products' basis of the Chebyshev sums (mray_amd/csrc/cheb_blocks.hpp)
against direct sums of cos(j theta) in extended precision, on the host, for
every width from 1 to 128 and angles including 0 and pi. An order's value is an
alternating sum of at most ceil(M / P) <= 13 products with one rounding each and
T_j's own error grows like j^2 u next to x = +-1 (u = 2^-53, j <= 127): the
bound is 2 * 127^2 u = 3.6e-12 of the terms' magnitudes."""
import pathlib
import shutil
import subprocess

import pytest

HERE = pathlib.Path(__file__).resolve().parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_products_basis_matches_direct_sums(tmp_path):
    exe = tmp_path / "chk"
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-Wno-unknown-pragmas", "-o", str(exe),
                    str(HERE / "cheb_blocks_check.cpp")], check=True)
    series, sums = map(float, subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split())
    print(f"series {series:.2e}, sums {sums:.2e}")
    assert series <= 3.6e-12
    assert sums <= 3.6e-12
