"""The FP64 tables of the matrix-core x and y lines: their error repeats on
every z-slice, so what counts is that of the table itself, not of the
arithmetic.  Against the exact operator with the same phases, in long double.

Bound: entries of M - c of at most |e|/n1 (e the largest increment, up to 2)
rounded once to 53 bits, relative to the field 2 * 2^-53 * 0.41 (the rms of a
rounding over a binade) = 9e-17.  Roots of unity and sums in double gave
2.1e-16 on 128 points."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def results(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("emu") / "dense_tables")
    subprocess.run([gxx, "-O2", "-std=c++17", "-I", os.path.join(HERE, "emu", "include"), "-o", exe,
                    os.path.join(HERE, "emu", "dense_tables.cpp")], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    return {ln.split()[0]: float(ln.split()[1]) for ln in out.strip().splitlines()}


@pytest.mark.parametrize("case", ["slice_16", "slice_32", "slice_64", "slice_96", "slice_128", "absorbing_96", "space_64",
                                  "space_128"])
def test_table(results, case):
    print(case, results[case])
    assert results[case] < 9e-17, (case, results[case])
