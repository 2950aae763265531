"""The entropy decoder's choice of a symbol by lanes (mray_amd/csrc/fastac_lanes.hpp),
compiled for the host, against the reference's bisection: random codes, whose
symbols and intervals must be the same bits, and malformed ones of 0xFF bytes,
whose value leaves the interval and goes to infinity after more than a million
symbols. There every lane past the alphabet must still be refused: a symbol of
64 lanes' worth would index past the model's counts."""
import pathlib
import shutil
import subprocess

import pytest

HERE = pathlib.Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    exe = tmp_path_factory.mktemp("fastac") / "chk"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-Wno-unknown-pragmas", "-o", str(exe),
                    str(HERE / "fastac_lanes_check.cpp")], check=True)

    def run(bits, byte, n):
        out = subprocess.run([str(exe), str(bits), str(byte), str(n)], check=True, capture_output=True, text=True)
        return [int(v) for v in out.stdout.split()]

    return run


@pytest.mark.parametrize("bits", range(1, 9))
def test_random_codes(check, bits):
    assert check(bits, -1, 200000) == [-1, 0]


@pytest.mark.parametrize("bits,n", [(5, 1400000), (4, 3900000), (7, 400000), (8, 300000)])
def test_codes_that_leave_the_interval(check, bits, n):
    first, infinite = check(bits, 255, n)
    assert first == -1, f"symbol {first} differs from the reference's"
    assert infinite
