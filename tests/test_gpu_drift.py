"""FP64 links whose rounding has drifted: the forms that take a link's adjoint for its inverse leave them
to the forms that do not.
"""
import ctypes

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def FL():
    import flue_lat_amd as FL
    return FL


@pytest.mark.parametrize("dims", [(3, 16, 16, 32), (11, 20, 21, 23)])
def test_magnetic_of_drifted_links(FL, dims):
    # Links 1.5e-14 longer than unitary: a leaf moved along them by their adjoints instead of their inverses
    # is 3e-14 too long for each link.  By quadrants nothing moves; their sums of positive terms round some
    # 1e-15 apart.
    f = FL.GaugeField.random(dims, 5, 0.3, "fp64")
    f.data.mul_(1.0 + 1.5e-14)
    ref = f.magnetic(variant=4)
    for v in (0, 7):
        assert abs(f.magnetic(variant=v) - ref) < 1e-14 * ref


@pytest.mark.parametrize("mu,nu", [(2, 1), (3, 4), (1, 3)])
def test_fmunu_of_drifted_links(FL, mu, nu):
    # by quadrants, as without a workspace: the same numbers
    from flue_lat_amd import _lib
    f = FL.GaugeField.random((12, 13, 31, 20), 9, 0.3, "fp64")
    f.data.mul_(1.0 + 1.5e-14)
    want = torch.empty_like(f.fmunu(mu, nu))
    st = (ctypes.c_int64 * 6)(*want.stride())
    _lib.check(_lib.lib().flue_fmunu(f._cdims, ctypes.c_void_p(f.data.data_ptr()), f.prec, mu, nu, 0,
                                     ctypes.c_void_p(want.data_ptr()), _lib.FLUE_OUT_STRIDED, st,
                                     ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "flue_fmunu")
    assert torch.equal(f.fmunu(mu, nu), want)


@pytest.mark.parametrize("dims", [(7, 24, 24, 23), (9, 20, 22, 24), (2, 34, 33, 47), (1, 400, 15, 16), (3, 16, 16, 16)])
def test_magnetic_of_a_field_that_is_not_unitary(FL, dims):
    # every link scaled: blocks of the quadrant form dealt to more partials than there are blocks, and to
    # fewer.  Against the quadrant form: the same numbers in sums of another order; an ensemble likewise.
    from flue_lat_amd.ensemble import Ensemble
    e = Ensemble.random([dims, (13, 14, 17, 33), dims], [5, 6, 7], 0.3, "fp64")
    e.data.mul_(1.01)
    ref = [e.field(c).magnetic(variant=4) for c in range(3)]
    for v in (0, 7):
        assert abs(e.field(0).magnetic(variant=v) - ref[0]) < 1e-14 * ref[0]
    _, B = e.flow(0.01, 0, measure_every=1)
    for c in range(3):
        assert abs(B[0, c] - ref[c]) < 1e-14 * ref[c]
