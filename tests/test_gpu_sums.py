"""Lattice sums are compensated across the groups of sites that a block adds up.

Links that are multiples of 1 make a Wilson loop a product of numbers chosen here.  All are powers of two,
so every loop is exact, and each row of 16 sites has one value; rows of 2^60 and -2^60 cancel and leave
rows of 2^-20, which a plain sum of the block loses.  The sum is then exact but for the division by the
volume.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

BIG, SMALL = 2.0 ** 30, 2.0 ** -10


@pytest.fixture(scope="module")
def FL():
    import flue_lat_amd as FL
    return FL


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("size", [1, 3])     # tables of one loop and of three by three
@pytest.mark.parametrize("minus", [5, 9])    # the row that cancels row 1
def test_wilson_loop_blocks_are_compensated(FL, prec, size, minus):
    dims = (2, 16, 16, 3)
    s = np.zeros(16)
    s[1] = s[2] = s[minus] = BIG
    s[minus + 1] = -BIG
    s[8:] = SMALL if minus == 5 else s[8:]
    if minus == 9:
        s[4:8] = s[12:] = SMALL
    rows = s * np.roll(s, -1)                # a 1 x 1 loop of the plane (x, y) at row y
    assert rows.max() == 2.0 ** 60 and rows.min() == -2.0 ** 60
    left = rows[np.abs(rows) < 1.0].sum()
    assert left == (7 if minus == 5 else 6) * 2.0 ** -20
    U = np.zeros(dims + (4, 3, 3), dtype=np.complex128)
    U[..., :, :, :] = np.eye(3)
    U[:, :, :, :, 1] *= s[None, None, :, None, None, None]
    f = FL.GaugeField.from_complex(U, prec, check=False)
    want = 3.0 * left / 16
    assert abs(f.wilson_loops(2, 3, size, size)[0, 0] - want) < 1e-15 * want
    got = f.wilson_loops_slices(2, 3, size, size)[0, 0]
    assert np.abs(got - want).max() < 1e-15 * want
    assert abs(f.wilson_loops(3, 2, size, size)[0, 0] - want) < 1e-15 * want
