"""The rule of which rays the gridded march of generate takes
(mray_amd/csrc/march_grid.hpp), compiled for the host: every ray it takes is
marched to its end, in increments within 2^-11 of the step (half of the
distance of floats at 8192 steps from t = 0, the rule's reach), also from
far behind the camera (a negative znear), where t + s no longer advances."""
import pathlib
import shutil
import subprocess

import pytest

HERE = pathlib.Path(__file__).resolve().parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_gridded_rays_end_in_uniform_steps(tmp_path):
    exe = tmp_path / "chk"
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-o", str(exe),
                    str(HERE / "march_grid_check.cpp")], check=True)
    taken, endless, worst = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()
    assert int(taken) > 10000
    assert int(endless) == 0, f"{endless} of {taken} gridded rays have no end"
    assert float(worst) <= 2.0 ** -11
