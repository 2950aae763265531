"""The gridded march of generate (mray_amd/csrc/march_grid.hpp), compiled for the
host. Its rule: every ray it takes is marched to its end, in increments within
2^-11 of the step (half of the distance of floats at 8192 steps from t = 0, the
rule's reach), also from far behind the camera (a negative znear), where t + s
no longer advances. Its weights: moments against the reference's integral in
long double, next to the rule's reach, where the steps of t change most and
the segments overlap most."""
import pathlib
import shutil
import subprocess

import pytest

HERE = pathlib.Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    exe = tmp_path_factory.mktemp("march_grid") / "chk"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-Wno-unknown-pragmas", "-o", str(exe),
                    str(HERE / "march_grid_check.cpp")], check=True)
    return lambda *args: subprocess.run([str(exe), *args], check=True, capture_output=True, text=True).stdout.split()


def test_gridded_rays_end_in_uniform_steps(check):
    taken, endless, worst = check()
    assert int(taken) > 10000
    assert int(endless) == 0, f"{endless} of {taken} gridded rays have no end"
    assert float(worst) <= 2.0 ** -11


def test_moments_next_to_the_reach(check):
    """2^-25 is half a unit of a float moment in [1/4, 1/2): what the rounding to
    float that follows costs."""
    worst, changes = check("300")
    print(f"largest error {worst}, {changes} rays whose increment changes")
    assert int(changes) > 20
    assert float(worst) <= 2.0 ** -25
