"""The FP32 matrix-core line operator compiled for the host, in the kernels'
order of operations and with the constant that they add.

drift: 100 slices against FP64, a random walk of 1.5e-7 a slice, to 2e-6.
Residuals of the table entries set to zero give 2.5e-6 on drift_beam_128 and
drift_noise_256 and a gain of 1e-9 to 3e-9 everywhere; a table that leaves out
what the constant misses of 1/12 fails by orders of magnitude.
gain: the mean change of the power in a slice over 6e7 complex values, four
standard deviations of unbiased roundings, 4 * 2 * 1.5e-7 / sqrt(1.2e8) = 1.1e-10;
with 1/12 rounded to FP32 as the constant the 96-point lines lose 2.4e-10."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
BOUND = {"drift": 2e-6, "gain": 1.1e-10}


@pytest.fixture(scope="module")
def results(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("emu") / "dense_product")
    subprocess.run([gxx, "-O2", "-march=native", "-ffp-contract=off", "-std=c++17", "-I",
                    os.path.join(HERE, "emu", "include"), "-o", exe, os.path.join(HERE, "emu", "dense_product.cpp")],
                   check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    return {ln.split()[0]: float(ln.split()[1]) for ln in out.strip().splitlines()}


@pytest.mark.parametrize("case", ["drift_beam_32", "drift_beam_64", "drift_beam_96", "drift_beam_128", "drift_noise_96",
                                  "drift_noise_128", "drift_noise_256", "gain_64", "gain_96", "gain_128"])
def test_dense_product(results, case):
    print(case, results[case])
    assert abs(results[case]) < BOUND[case.split("_")[0]], (case, results[case])
