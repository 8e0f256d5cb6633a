"""The dk phase on grids with pixels, which takes variant 0 of the time pass
(the register form for 512 and 1024 samples) with arguments of its own per
slice: two trips with modulator, GDD and free space against the FP64 oracle,
fields to 1e-5 in FP32 (about 2e-7 per slice as a random walk) and 1e-11 in
FP64, as for the plane wave."""
import pytest

import cuopo3d_amd as co
from cuopo3d_amd import configs
from cuopo3d_amd.capi import OPO_FP32, OPO_FP64
from oracle.pyoracle import Oracle

from helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,prec", [((16, 16, 64), OPO_FP32), ((16, 16, 256), OPO_FP32), ((16, 16, 512), OPO_FP32),
                                    ((32, 16, 512), OPO_FP32), ((16, 16, 1024), OPO_FP32), ((16, 16, 2048), OPO_FP32),
                                    ((16, 16, 256), OPO_FP64), ((16, 16, 1024), OPO_FP64)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_trips_with_dk_phase(n, prec, require_gpu):
    grid, p, ph, fields = configs.cavity_64(n=n, n_round_trips=3, precision=prec)
    p.n_slices = 7
    p.dk, p.dk_phase_scale = 1e-2, 1.0
    p.eom_on, p.eom_beta, p.eom_fpm = 1, 0.5, 2.0 / p.t_window
    o = Oracle(grid, p)
    o.set_fields(*fields)
    o.run_round_trips(2)
    with co.Solver(grid, p, device=0) as s:
        s.set_fields(*fields)
        s.runOPO(2)
        errs = [rel_l2(a, b) for a, b in zip(s.get_fields(), o.get_fields())]
    print(n, prec, errs, flush=True)
    assert max(errs) < (1e-5 if prec == OPO_FP32 else 1e-11), errs
