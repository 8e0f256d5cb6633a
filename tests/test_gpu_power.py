"""Signal power of FP32 cavities against the FP64 path on the same inputs (its
own error is 1e-14 per trip).  Random rounding errors average out over the
cells; a gain that an operator leaves adds up over the slices.  Bound: 6e-11
per slice, so 1e-6, the per-trip power target, holds for 160 trips of 100
slices.  A residual lost in the dispersion table's product left 1.2e-10 per
slice on 64 x 64 x 256 (1.3e-10 on 32 x 32 x 128), and 1/12 in FP32 as the
constant of the 96-point lines 7e-10 on 96 x 96 x 128."""
import numpy as np
import pytest

import cuopo3d_amd as co
from cuopo3d_amd import configs
from cuopo3d_amd.capi import OPO_FP32, OPO_FP64

pytestmark = pytest.mark.gpu

TRIPS = 30


@pytest.mark.parametrize("n", [(64, 64, 256), (128, 128, 64), (96, 96, 128)], ids=lambda n: "x".join(map(str, n)))
def test_signal_power_has_no_gain(n, require_gpu):
    power = {}
    for prec in (OPO_FP64, OPO_FP32):
        grid, p, ph, fields = configs.cavity_64(n=n, n_round_trips=200, precision=prec)
        fields = [f.astype(np.complex64) for f in fields]   # the same values in both
        with co.Solver(grid, p, device=0) as s:
            s.set_fields(*[f.astype(np.complex128) if prec == OPO_FP64 else f for f in fields])
            power[prec] = s.runOPO(TRIPS)[:, 1]
    err = power[OPO_FP32] / power[OPO_FP64] - 1
    gain = (err[-1] - err[0]) / ((TRIPS - 1) * p.n_slices)
    print(n, f"error after one trip {err[0]:.2e}, {TRIPS} trips {err[-1]:.2e}, per slice {gain:.2e}", flush=True)
    assert abs(gain) < 6e-11, gain
    assert abs(err[0]) < 1e-6
