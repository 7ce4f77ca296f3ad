"""Tuning the plaquette of a small lattice does not replace its untuned form by a slower one."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_tuning_leaves_the_faster_untuned_plaquette(prec, tmp_path):
    # 8^3x16: a thread per site and plane takes two thirds of the time of the shortest walk.  An older choice
    # is dropped too.
    import flue_lat_amd as FL
    from flue_lat_amd import _lib
    dims = (16, 8, 8, 8)
    f = FL.GaugeField.random(dims, 3, 0.3, prec)
    before = f.plaquette()[0]
    table = tmp_path / "tune.txt"
    table.write_text(f"0 2 {f.prec} 16 8 8 8 4 1.0\n")
    FL.field.tune_load(table)
    v, ms = f.autotune("plaquette", reps=200)
    assert 1 <= v <= 6 and ms > 0
    tuned = ctypes.c_int32(-1)
    _lib.check(_lib.lib().flue_tuned_variant(_lib.OPS["plaquette"], f._cdims, f.prec, ctypes.byref(tuned)),
               "flue_tuned_variant")
    assert tuned.value == 0
    assert f.plaquette()[0] == before
