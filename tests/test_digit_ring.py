"""The arithmetic encoder's digit ring (mray_amd/csrc/digit_ring.hpp), compiled
for the host with 64 emulated lanes, against bytes written and carried one by
one as the reference does: runs of 0xFFFF of 0 to 200 digits with a carry behind
them at every offset around a flush (so that carries leave the flushed group for
bytes already out and ripple there, which ordinary data meets once in 2^16
flushes), random digits and carries, and codes cut off at their capacity."""
import pathlib
import shutil
import subprocess

import pytest

HERE = pathlib.Path(__file__).resolve().parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_digits_and_carries(tmp_path):
    exe = tmp_path / "chk"
    subprocess.run(["g++", "-O1", "-std=c++17", "-o", str(exe), str(HERE / "digit_ring_check.cpp")], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()
    sequences, bad, late, rounds = map(int, out)
    assert bad == 0, f"{bad} of {sequences} codes differ"
    # the paths that this is about were taken
    assert late > 1000 and rounds > 1000
