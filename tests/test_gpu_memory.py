"""Calls whose fast forms take a workspace of the size of the field run without room for it."""
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_magnetic_and_fmunu_without_room_for_footprints(monkeypatch, prec):
    import flue_lat_amd as FL
    f = FL.GaugeField.random((12, 25, 34, 31), 3, 0.3, prec)   # ragged, and large enough for the tiles
    B, F = f.magnetic(), f.fmunu(2, 3)
    g = f.clone()
    empty = torch.empty

    def full(*args, **kw):
        if kw.get("dtype") is torch.uint8 and args[0] > 32 << 20:
            raise torch.cuda.OutOfMemoryError("no room")
        return empty(*args, **kw)

    monkeypatch.setattr(torch, "empty", full)
    assert abs(g.magnetic() - B) < (1e-12 if prec == "fp64" else 1e-6) * B
    got = g.fmunu(2, 3)
    monkeypatch.undo()
    assert float((got - F).abs().max()) < (1e-13 if prec == "fp64" else 2e-6) * float(F.abs().max())
    assert g.magnetic() == B   # with room again
