"""FP64 planes with few lines, which run in LDS bands instead of whole lines per
wave: sizes on both sides of the rule, against the FP64 oracle on random
fields.  1e-13 relative L2 per operator pair as for the matrix-core planes
(about 40 roundings of two transform pairs); diffraction alone, the large
phases of free space being limited by their FP64 argument."""
import pytest

import cuopo3d_amd as co
from cuopo3d_amd.capi import OPO_FP64
from oracle.pyoracle import Oracle

from helpers import cavity_params, random_fields, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(64, 96, 1), (64, 128, 1), (128, 64, 1), (96, 128, 1), (128, 96, 1), (128, 128, 1),
                               (128, 32, 1), (128, 128, 16), (96, 96, 1), (64, 256, 1), (96, 256, 16), (128, 256, 16),
                               (96, 256, 32), (256, 128, 1), (256, 128, 16), (512, 128, 1), (128, 512, 1),
                               (512, 512, 1)], ids=lambda n: "x".join(map(str, n)))
def test_few_lines(n, require_gpu):
    grid, p, _ = cavity_params(n, precision=OPO_FP64, t_window=20.0)
    fields = random_fields(grid, sum(n), precision=OPO_FP64)
    o = Oracle(grid, p)
    o.set_fields(*fields)
    o.diffraction()
    with co.Solver(grid, p, device=0) as s:
        s.set_fields(*fields)
        s.diffractionInCrystal()
        errs = [rel_l2(a, b) for a, b in zip(s.get_fields(), o.get_fields())]
    print(n, errs, flush=True)
    assert max(errs) < 1e-13, errs
