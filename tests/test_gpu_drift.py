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
