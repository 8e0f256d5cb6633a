"""Stage times of plane-wave solves in a batch: one t-pass launch per trip over
all of them, so its algorithmic bytes are those of all of them also where their
slice counts differ, in both ways of timing."""
import pytest

import cuopo3d_amd as co
from cuopo3d_amd import configs
from cuopo3d_amd.capi import OPO_FP32, OPO_FP64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [OPO_FP32, OPO_FP64], ids=["fp32", "fp64"])
def test_plane_wave_launch_bytes(prec, require_gpu):
    b = co.Batch(1 << 28, prec)
    for slices in (9, 5):
        grid, p, _, fields = configs.cavity_64(n=(1, 1, 256), n_round_trips=8, precision=prec)
        p.no_diffraction, p.n_slices = 1, slices
        b.submit(grid, p, *fields, 8)
    b.step()
    b.profile(True)
    b.step()          # re-captured with the event nodes
    b.profile(True)   # sums back to zero
    b.step()
    try:
        read = b.profile_read()
    except RuntimeError as e:   # a runtime that cannot time graph event nodes
        print("in-graph event timing unavailable:", e, flush=True)
        read = None
    b.profile(False)
    timed = b.time_stages(reps=2)
    b.close()
    want = 2 * 256 * (96 if prec == OPO_FP64 else 48)
    for entries, launches in ((read, 1), (timed, 2)):
        if entries is not None:
            got = [(e["size"], e["launches"], e["alg_bytes"]) for e in entries if e["stage"] == "time_op"]
            print(got, flush=True)
            assert got == [(-256, launches, want)], got
