"""Tile-shape cache of the autotuner (host side, no device needed)."""
import ctypes as C

import pytest

import uir

SPEC = dict(n=128, n_dets=182, n_angles=90, step=0.0349066, relaxation=0.5)


def test_untuned_geometry_gets_the_default_shape():
    uir.tune_clear()
    tile, tuned = uir.tune_get(SPEC, "f16")
    assert not tuned and tile == {"fp_angles": 16, "bp_angles": 32, "bp_rows": 64}


def test_set_get_per_geometry_and_dtype():
    uir.tune_clear()
    uir.tune_set(SPEC, "f16", 8, 16, 32)
    assert uir.tune_get(SPEC, "f16") == ({"fp_angles": 8, "bp_angles": 16, "bp_rows": 32}, True)
    assert uir.tune_get(SPEC, "f32")[1] is False                     # dtype is part of the key
    assert uir.tune_get(dict(SPEC, n_angles=91), "f16")[1] is False  # so is the geometry
    uir.tune_set(SPEC, "f16", 16, 32, 32)                            # overwrite
    assert uir.tune_get(SPEC, "f16")[0]["bp_rows"] == 32
    uir.tune_clear()
    assert uir.tune_get(SPEC, "f16")[1] is False


@pytest.mark.parametrize("tile", [(12, 32, 64), (64, 32, 64), (16, 8, 64), (16, 32, 48), (0, 0, 0)])
def test_only_built_variants_are_accepted(tile):
    with pytest.raises(uir.UirError) as e:
        uir.tune_set(SPEC, "f16", *tile)
    assert e.value.status == 1


class _Tile(C.Structure):
    _fields_ = [(k, C.c_int32) for k in ("fp_angles", "bp_angles", "bp_rows", "fp_single", "bp_tuned")]


class _Choice(C.Structure):
    _fields_ = [(k, C.c_int) for k in ("pairs", "rows32", "angles16")]


@pytest.mark.parametrize("tuned", [None, (16, 32, 64), (16, 16, 64), (16, 32, 32)])
def test_tuned_bp_shape_keeps_its_angles(tuned):
    """The rule on slice pairs sets the staged angles of an untuned geometry
    only, also where tuning measured the default shape as the fastest."""
    L = uir.load()
    L.uir_tile_for.restype = L.uirk_plan_bp_tile.restype = _Tile
    L.uirk_plan_bp_tile.argtypes = [_Tile, _Choice, C.c_int]
    uir.tune_clear()
    if tuned:
        uir.tune_set(SPEC, "f16", *tuned)
    spec = uir.slice_spec(SPEC)
    tile = L.uir_tile_for(C.byref(spec), uir.DTYPE_F16)
    got = L.uirk_plan_bp_tile(tile, _Choice(1, 0, 1), 0)
    assert (got.bp_angles, got.bp_rows) == (tuned[1:] if tuned else (16, 64))
    got = L.uirk_plan_bp_tile(tile, _Choice(1, 1, 0), 0)
    assert (got.bp_angles, got.bp_rows) == (tuned[1] if tuned else 32, 32)
    uir.tune_clear()
