"""The admission footprint of a batched solve counts its table block as it is
allocated: rotations (4 n elements of x and y together) for lines in LDS, none
for lines on the matrix cores; five x and five y tables of 2 n elements (FP32
matrix-core sizes 3 n); rotations, D, GDD and modulator tables of the time axis,
12 NT; every allocation in units of 64 KiB."""
import ctypes as C

import pytest

from cuopo3d_amd import capi
from cuopo3d_amd.capi import Grid, OPO_FP32, OPO_FP64

UNIT = 65536


def _units(b):
    return -(-b // UNIT) * UNIT


def _table_elements(n, nt, fp64):
    size = n in (16, 32, 64, 96, 128) or (n == 256 and not fp64)   # has a matrix-core form
    used = size and (n < 256 or nt * n >= 16 * 256)
    return (0 if used else 4 * n) + 10 * (3 * n if size and not fp64 else 2 * n) + 12 * nt


@pytest.mark.parametrize("prec", [OPO_FP32, OPO_FP64], ids=["fp32", "fp64"])
@pytest.mark.parametrize("n", [1, 16, 32, 64, 96, 128, 256, 512])
def test_footprint_covers_the_tables(n, prec):
    lib = capi.load()
    fp64 = prec == OPO_FP64
    cb = 16 if fp64 else 8
    for nt in (16, 32, 64, 128, 256, 512, 1024, 2048) + (() if fp64 else (4096,)):
        cells = n * n * nt
        blocks = min(max(-(-cells // 4096), 1), 1024)
        want = (4 * _units(cells * cb) + _units(_table_elements(n, nt, fp64) * cb) + _units(8 * (3 * blocks + 4)) + UNIT
                + _units(24 * 7))
        got = lib.opo_batch_footprint(C.byref(Grid(n, n, nt)), prec, 7)
        assert got == want, (n, nt, got - want)
