"""Complex arrays of any element order into a field and back.

Three kernels serve three kinds of order (sites contiguous, x fastest, another direction
fastest) and a general one the rest, so the orders here mix them with extents of 1, extents past a
tile's edge, expanded (zero-stride) sources and a pointer that is not aligned to its element.  A
conversion moves values, so results are compared exactly (FP32: the rounded value).
"""
import ctypes
import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# memory orders, slowest axis first, of the axes (t, x, y, z, mu, a, b)
ORDERS = [(0, 1, 2, 3, 4, 5, 6), (6, 5, 4, 3, 2, 1, 0), (4, 5, 6, 0, 3, 2, 1), (0, 3, 2, 1, 4, 5, 6),
          (3, 2, 1, 0, 6, 4, 5), (4, 0, 1, 2, 5, 6, 3), (5, 6, 4, 1, 3, 0, 2), (0, 4, 1, 5, 2, 6, 3), (1, 0, 2, 4, 3, 6, 5)]
DIMS = [(5, 7, 6, 9), (1, 3, 2, 1), (3, 70, 2, 5), (37, 1, 3, 40), (2, 33, 35, 1)]


@pytest.fixture(scope="module")
def FL():
    import flue_lat_amd as FL
    return FL


def ordered(U, order):
    """U with its axes in the given memory order"""
    inv = [order.index(k) for k in range(7)]
    return U.permute(order).contiguous().permute(inv)


def planes(U):
    return torch.view_as_real(U.permute(4, 5, 6, 0, 3, 2, 1).contiguous()).reshape(-1)


@pytest.mark.parametrize("cdtype", [torch.complex128, torch.complex64])
@pytest.mark.parametrize("dims", DIMS)
def test_every_order(FL, dims, cdtype):
    from flue_lat_amd import _lib
    lib, st = _lib.lib(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    torch.manual_seed(sum(dims))
    U = torch.randn(dims + (4, 3, 3), dtype=cdtype, device="cuda")
    code = _lib.FLUE_C64 if cdtype == torch.complex64 else _lib.FLUE_C128
    for order in ORDERS:
        A = ordered(U, order)
        for prec, dt in (("fp64", torch.float64), ("fp32", torch.float32)):
            f = FL.GaugeField.from_complex(A, prec, check=False)
            assert torch.equal(f.data, planes(U).to(dt)), (order, prec)
            out = torch.zeros_like(A)   # keeps A's strides
            assert out.stride() == A.stride()
            rc = lib.flue_export_field(f._cdims, ctypes.c_void_p(f.data.data_ptr()), f.prec, ctypes.c_void_p(out.data_ptr()),
                                       code, (ctypes.c_int64 * 7)(*out.stride()), st)
            assert rc == 0
            want = U.to(torch.complex64).to(cdtype) if prec == "fp32" else U
            assert torch.equal(out, want), (order, prec)


def test_expanded_and_unaligned_sources(FL):
    from flue_lat_amd import _lib
    dims = (4, 6, 5, 3)
    one = torch.randn((1, 1, 1, 1, 4, 3, 3), dtype=torch.complex128, device="cuda")
    E = one.expand(dims + (4, 3, 3))
    assert torch.equal(FL.GaugeField.from_complex(E).data, planes(E))
    # a complex128 array that starts 8 bytes past a 16-byte boundary, in and out
    U = torch.randn(dims + (4, 3, 3), dtype=torch.complex128, device="cuda")
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    cs = (ctypes.c_int64 * 7)(*U.stride())
    buf = torch.zeros(2 * U.numel() + 1, dtype=torch.float64, device="cuda")
    buf[1:] = torch.view_as_real(U).reshape(-1)
    f = FL.GaugeField(dims)
    ptr = ctypes.c_void_p(buf.data_ptr() + 8)
    assert _lib.lib().flue_import_field(f._cdims, ptr, _lib.FLUE_C128, cs, ctypes.c_void_p(f.data.data_ptr()), 0, st) == 0
    assert torch.equal(f.data, planes(U))
    buf.zero_()
    assert _lib.lib().flue_export_field(f._cdims, ctypes.c_void_p(f.data.data_ptr()), 0, ptr, _lib.FLUE_C128, cs, st) == 0
    assert torch.equal(buf[1:], torch.view_as_real(U).reshape(-1)) and buf[0] == 0


@pytest.mark.parametrize("dims", [(3, 5, 7, 6), (1, 17, 2, 4), (2, 16, 3, 9), (4, 1, 1, 1)])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_tangent_field(FL, dims, prec):
    # 2 G U against the product of the exported arrays: one rounding per product and sum of three
    # (6 eps relative to the row norms)
    from flue_lat_amd.autograd import _tangent, tangent_from_lie
    g = FL.GaugeField.random(dims, 31, 0.3, "fp64")
    U = g.to_complex()
    f = g.astype(prec)
    G = f.wilson_grad(6.0)
    E = _tangent(G, U, f)
    assert E.is_contiguous() and E.shape == dims + (4, 3, 3)
    want = tangent_from_lie(G.to_complex(), U)
    assert float((E - want).abs().max()) <= 6 * 2.3e-16 * 2 * float(want.abs().max())


@pytest.mark.parametrize("dims", [(3, 1, 1, 1), (4, 1, 3, 1), (3, 4, 1, 2), (5, 7, 3, 4), (1, 1, 1, 2), (33, 34, 3, 2)])
def test_host_functions_copy_what_they_read(FL, dims):
    # the host functions bring the directions they read to the device; the same kernels on a resident
    # field of all of them give the same numbers
    fc = FL.compiled.flue_c
    U = np.asfortranarray(FL.GaugeField.random(dims, 17, 0.4).to_complex().cpu().numpy())
    f = FL.GaugeField.from_complex(U)
    for args in itertools.product(range(1, 5), range(1, 5), range(1, 5)):
        assert fc.plaquette_c(U, *args)[:2] == f.plaquette(*args), args
    if dims[0] >= 3:
        assert fc.polyakov_c(U)[:2] == f.polyakov()
    assert fc.magnetic_c(U) == f.magnetic()
    for mu, nu in itertools.product(range(1, 5), range(1, 5)):
        assert np.array_equal(fc.loop5munucoord_c(U, mu, nu), f.fmunu(mu, nu).cpu().numpy())
        assert fc.wmunu_c(U, mu, nu, 2, 1) == f.wilson_loop(mu, nu, 2, 1)
        assert fc.wmunutau_c(U, 1, mu, nu, 1, 2) == f.wilson_loop(mu, nu, 1, 2, tau=1)


def test_host_functions_copy_two_and_three_directions(FL):
    # 18,018 sites: leaving out a single direction saves more than the 2 MB from which a part of the array is
    # copied, so every call that reads two or three directions takes them out of the array by rows
    dims = (14, 9, 11, 13)
    fc = FL.compiled.flue_c
    U = np.asfortranarray(FL.GaugeField.random(dims, 17, 0.4).to_complex().cpu().numpy())
    f = FL.GaugeField.from_complex(U)
    for args in ((1, 4, 4), (2, 4, 4), (1, 1, 4), (1, 3, 3), (2, 3, 3), (3, 3, 4), (1, 2, 2), (2, 2, 4)):
        assert fc.plaquette_c(U, *args)[:2] == f.plaquette(*args), args
        assert fc.genplaquette_c(U, *args)[:2] == f.plaquette(*args), args
    assert fc.polyakov_c(U)[:2] == f.polyakov()
    assert fc.magnetic_c(U) == f.magnetic()
    for mu, nu in itertools.product(range(1, 5), range(1, 5)):
        assert np.array_equal(fc.loop5munucoord_c(U, mu, nu), f.fmunu(mu, nu).cpu().numpy()), (mu, nu)
        assert np.array_equal(fc.cloverloopmunucoord_c(U, mu, nu), f.fmunu(mu, nu, clover=True).cpu().numpy()), (mu, nu)
        assert fc.wmunu_c(U, mu, nu, 2, 1) == f.wilson_loop(mu, nu, 2, 1), (mu, nu)
        assert fc.wmunutau_c(U, 3, mu, nu, 1, 2) == f.wilson_loop(mu, nu, 1, 2, tau=3), (mu, nu)
