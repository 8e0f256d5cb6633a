"""No systematic gain in the FP32 operators, compiled for the host: a bias of
the power by rounding adds up linearly over the z-slices of a cavity, where
random errors do not.

Bounds: five standard deviations of the mean over 4e6 random values of
unbiased roundings, whose error is 6e-8 (one product) or 2e-7 (an operator)
relative to the value: 2 * 6e-8 / sqrt(4e6) * 5 = 3e-10 and 1e-9.  A residual
of a table entry that is added to the larger product is lost in its rounding:
5e-9 and 4e-9 with the phases of a dispersion slice."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
BOUND = {"mul": 3e-10, "line": 1e-9}


@pytest.fixture(scope="module")
def results(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("emu") / "gain")
    subprocess.run([gxx, "-O2", "-std=c++17", "-I", os.path.join(HERE, "emu", "include"), "-o", exe,
                    os.path.join(HERE, "emu", "gain.cpp")], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    return {ln.split()[0]: float(ln.split()[1]) for ln in out.strip().splitlines()}


@pytest.mark.parametrize("case", ["mul_1e-4", "mul_5e-4", "mul_1e-3", "mul_0.3", "mul_2.8", "mul_absorbing", "line_64",
                                  "line_256", "line_2048"])
def test_no_gain(results, case):
    print(case, results[case])
    assert abs(results[case]) < BOUND[case.split("_")[0]], (case, results[case])
