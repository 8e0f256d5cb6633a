"""Launch-variant tables as host state (no GPU): what opo_tune_get returns can
be given back to opo_tune_set, and the state is then what it was, also where
nothing was chosen and the choice goes by the pixels of the work (-1)."""
import pytest

from cuopo3d_amd import capi
from cuopo3d_amd.capi import OPO_FP32, OPO_FP64, OPO_TUNE_TIME_PASS, OPO_TUNE_XY_PASS

NT = (1, 16, 32, 64, 128, 256, 512, 1024, 2048, 4096)
NX = (1, 16, 32, 64, 96, 128, 256, 512)


def _entries():
    for prec in (OPO_FP32, OPO_FP64):
        for n in NT:
            if n < 4096 or prec == OPO_FP32:
                yield prec, OPO_TUNE_TIME_PASS, n
        for n in NX:
            yield prec, OPO_TUNE_XY_PASS, n


@pytest.mark.parametrize("prec,axis,n", list(_entries()))
def test_saved_choice_can_be_put_back(prec, axis, n):
    lib = capi.load()
    saved = lib.opo_tune_get(prec, axis, n)
    assert lib.opo_tune_set(prec, axis, n, -1) == capi.OPO_OK   # nothing chosen
    untuned = lib.opo_tune_get(prec, axis, n)
    try:
        for v in range(64):
            if lib.opo_tune_set(prec, axis, n, v) == capi.OPO_OK:
                assert lib.opo_tune_get(prec, axis, n) == v
                assert lib.opo_tune_set(prec, axis, n, untuned) == capi.OPO_OK
                assert lib.opo_tune_get(prec, axis, n) == untuned
    finally:
        assert lib.opo_tune_set(prec, axis, n, saved) == capi.OPO_OK
    assert lib.opo_tune_get(prec, axis, n) == saved


@pytest.mark.parametrize("prec,n", [(OPO_FP32, 64), (OPO_FP32, 256), (OPO_FP32, 512), (OPO_FP32, 1024),
                                    (OPO_FP32, 2048), (OPO_FP64, 64), (OPO_FP64, 256)])
def test_untuned_is_told_apart_from_a_choice(prec, n):
    """These time lines take another launch shape on few pixels than on many:
    no variant number stands for that."""
    lib = capi.load()
    saved = lib.opo_tune_get(prec, OPO_TUNE_TIME_PASS, n)
    assert lib.opo_tune_set(prec, OPO_TUNE_TIME_PASS, n, -1) == capi.OPO_OK
    assert lib.opo_tune_get(prec, OPO_TUNE_TIME_PASS, n) == -1
    assert lib.opo_tune_set(prec, OPO_TUNE_TIME_PASS, n, saved) == capi.OPO_OK


def test_no_entry_for_other_sizes():
    lib = capi.load()
    for axis, n in ((OPO_TUNE_TIME_PASS, 48), (OPO_TUNE_TIME_PASS, 8192), (OPO_TUNE_XY_PASS, 48), (OPO_TUNE_XY_PASS, 8)):
        assert lib.opo_tune_set(OPO_FP32, axis, n, -1) == capi.OPO_ERR_ARG
        assert lib.opo_tune_set(OPO_FP32, axis, n, 0) == capi.OPO_ERR_ARG
    assert lib.opo_tune_set(OPO_FP64, OPO_TUNE_TIME_PASS, 4096, -1) == capi.OPO_ERR_ARG   # FP32 only
    assert lib.opo_tune_set(OPO_FP32, OPO_TUNE_TIME_PASS, 256, -2) == capi.OPO_ERR_ARG


@pytest.mark.parametrize("prec,nx,accepted", [
    (OPO_FP32, 1, [0]), (OPO_FP32, 16, range(6)), (OPO_FP32, 32, range(6)), (OPO_FP32, 64, range(9)),
    (OPO_FP32, 96, [0, 1, 2, 7, 8]), (OPO_FP32, 128, [0, 1, 2, 7, 8]), (OPO_FP32, 256, range(3)), (OPO_FP32, 512, [0]),
    (OPO_FP64, 32, range(6)), (OPO_FP64, 64, range(3)), (OPO_FP64, 96, range(3)), (OPO_FP64, 128, range(3)),
    (OPO_FP64, 256, range(3)), (OPO_FP64, 512, [0])])
def test_xy_numbers_of_saved_choices_stay_valid(prec, nx, accepted):
    lib = capi.load()
    saved = lib.opo_tune_get(prec, OPO_TUNE_XY_PASS, nx)
    got = [v for v in range(-2, 64) if v != -1 and lib.opo_tune_set(prec, OPO_TUNE_XY_PASS, nx, v) == capi.OPO_OK]
    assert lib.opo_tune_set(prec, OPO_TUNE_XY_PASS, nx, saved) == capi.OPO_OK
    assert got == list(accepted)
