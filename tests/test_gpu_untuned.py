"""Untuned launch shapes: a tuner call that timed nothing chooses nothing, and
the shapes that a small and a large grid take by themselves give bitwise the
fields of variant 0."""
import re

import numpy as np
import pytest

import cuopo3d_amd as co
from cuopo3d_amd import configs
from cuopo3d_amd.capi import OPO_FP32, OPO_FP64, OPO_OK, OPO_TUNE_TIME_PASS, OPO_TUNE_XY_PASS

pytestmark = pytest.mark.gpu


@pytest.fixture
def untuned():
    """The time-pass entry of a size, untuned for the test."""
    lib = co.load()
    saved = {}

    def take(prec, nt):
        saved[prec, nt] = lib.opo_tune_get(prec, OPO_TUNE_TIME_PASS, nt)
        assert lib.opo_tune_set(prec, OPO_TUNE_TIME_PASS, nt, -1) == OPO_OK
        return lib

    yield take
    for (prec, nt), v in saved.items():
        assert lib.opo_tune_set(prec, OPO_TUNE_TIME_PASS, nt, v) == OPO_OK


@pytest.mark.parametrize("prec,nt", [(OPO_FP32, 256), (OPO_FP32, 2048), (OPO_FP64, 256)])
def test_tuner_on_a_plane_wave_chooses_nothing(prec, nt, untuned, require_gpu):
    """One pixel has no time-pass variants to time."""
    lib = untuned(prec, nt)
    grid, p, ph, fields = configs.cavity_64(n=(1, 1, nt), precision=prec)
    p.no_diffraction = 1
    with co.Solver(grid, p, device=0) as s:
        s.set_fields(*fields)
        report = s.autotune(reps=1)
    print(report, flush=True)
    assert lib.opo_tune_get(prec, OPO_TUNE_TIME_PASS, nt) == -1


@pytest.mark.parametrize("n", [(16, 16, 256), (64, 64, 256), (16, 16, 1024), (64, 64, 1024), (128, 128, 512),
                               (16, 16, 2048), (64, 64, 2048)], ids=lambda n: "x".join(map(str, n)))
def test_untuned_shapes_give_the_same_fields(n, untuned, require_gpu):
    lib = untuned(OPO_FP32, n[2])
    grid, p, ph, fields = configs.cavity_64(n=n, n_round_trips=4)
    p.n_slices = 3
    out = []
    for v in (-1, 0):
        assert lib.opo_tune_set(OPO_FP32, OPO_TUNE_TIME_PASS, n[2], v) == OPO_OK
        with co.Solver(grid, p, device=0) as s:
            s.set_fields(*fields)
            out.append((s.runOPO(2), *s.get_fields()))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("nx,prec,shapes", [(32, OPO_FP32, {0: 128, 3: 256, 4: 512, 5: 1024}), (64, OPO_FP32, {0: 256}),
                                            (96, OPO_FP32, {0: 384}), (64, OPO_FP64, {0: 256}),
                                            (256, OPO_FP64, {0: 256, 1: 512, 2: 256})])
def test_tuner_times_each_launch_shape_once(nx, prec, shapes, require_gpu):
    """Numbers that stand for the same launch are timed once, and the report
    gives the threads that run."""
    lib = co.load()
    keep = [(a, n, lib.opo_tune_get(prec, a, n)) for a, n in ((OPO_TUNE_TIME_PASS, 16), (OPO_TUNE_XY_PASS, nx))]
    grid, p, ph, fields = configs.cavity_64(n=(nx, nx, 16), precision=prec)
    try:
        with co.Solver(grid, p, device=0) as s:
            s.set_fields(*fields)
            report = s.autotune(reps=1)
    finally:
        for a, n, v in keep:
            assert lib.opo_tune_set(prec, a, n, v) == OPO_OK
    line = next(x for x in report.splitlines() if x.startswith(f"xy pass NX={nx}"))
    got = {int(v): int(b) for v, b in re.findall(r" v(\d+)\(tile \d+, block (\d+)", line)}
    assert got == shapes, line


def test_saved_persistent_choice_runs_the_plane_launch(require_gpu):
    """A number that stood for persistent workgroups gives the fields of variant
    0, alone and in a batch."""
    from helpers import batch_run
    lib = co.load()
    keep = lib.opo_tune_get(OPO_FP32, OPO_TUNE_XY_PASS, 64)
    grid, p, ph, fields = configs.cavity_64(n=(64, 64, 32), n_round_trips=2)
    out = []
    try:
        for v in (0, 8):
            assert lib.opo_tune_set(OPO_FP32, OPO_TUNE_XY_PASS, 64, v) == OPO_OK
            with co.Solver(grid, p, device=0) as s:
                s.set_fields(*fields)
                out.append((s.runOPO(2), *s.get_fields()))
            (res,), _ = batch_run([(grid, p, ph, fields)], 2)
            out.append((res[0], *res[1]))
    finally:
        assert lib.opo_tune_set(OPO_FP32, OPO_TUNE_XY_PASS, 64, keep) == OPO_OK
    for o in out[1:]:
        for a, b in zip(out[0], o):
            assert np.array_equal(a, b)
