"""Square and oblong cells on square planes: with dx = dy the y tables reuse what
the x tables computed, with dx != dy they must not.  Diffraction and free space
against the FP64 oracle on random fields.  Bounds: about 40 roundings per
operator pair (FP32 5e-7, FP64 1e-13), and in FP64 free space the rounding of
phases up to 3000 rad, a
few of 1.1e-16 each: 1e-12."""
import pytest

import cuopo3d_amd as co
from cuopo3d_amd.capi import OPO_FP32, OPO_FP64
from oracle.pyoracle import Oracle

from helpers import cavity_params, random_fields, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [OPO_FP32, OPO_FP64], ids=["fp32", "fp64"])
@pytest.mark.parametrize("dy", [1.0, 0.6], ids=["square", "oblong"])
@pytest.mark.parametrize("n", [16, 96, 128, 256])
def test_cells(n, dy, prec, require_gpu):
    grid, p, _ = cavity_params((n, n, 16), precision=prec, t_window=20.0)
    p.dy = dy * p.dx
    fields = random_fields(grid, n, precision=prec)
    o = Oracle(grid, p)
    with co.Solver(grid, p, device=0) as s:
        for gpu, ref, bound64 in ((s.diffractionInCrystal, o.diffraction, 1e-13),
                                  (s.diffractionInFreeSpace, o.free_space, 1e-12)):
            o.set_fields(*fields)
            ref()
            s.set_fields(*fields)
            gpu()
            errs = [rel_l2(a, b) for a, b in zip(s.get_fields(), o.get_fields())]
            print(n, dy, errs, flush=True)
            assert max(errs) < (5e-7 if prec == OPO_FP32 else bound64), errs
