"""Rectangle-first forms on extents that the tiles do not divide, against the oracle.

The tiles split an extent into nearly equal parts, so odd and prime extents leave tiles of two
widths, lanes idle in a tile's last turn, and transposes past an edge of 16.  Tolerances as for
the tileable lattices (tests/test_gpu_rect.py): FP64 sums 1e-12, FP32 links 1e-6; adjoint 1e-12
and 1e-5 of the largest entry.
"""
import ctypes

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# every extent below 16, none a multiple of it, primes, one row wider than a footprint
DIMS = [(39, 13, 14, 15), (5, 29, 27, 25), (3, 47, 17, 41), (2, 400, 12, 19)]


@pytest.fixture(scope="module")
def FL():
    import flue_lat_amd as FL
    return FL


@pytest.mark.parametrize("dims", DIMS)
def test_rect_uneven_extents(FL, dims):
    print(f"[tiles] {dims}", flush=True)
    U = O.random_field(dims, 8100 + dims[1], 0.3)
    want = O.magnetic(U)
    f = FL.GaugeField.from_complex(U)
    assert abs(f.magnetic(variant=7) - want) < 1e-12 * want
    assert f.magnetic() == f.magnetic(variant=7) == f.magnetic(variant=7)
    assert abs(f.astype("fp64-su3").magnetic(variant=7) - want) < 1e-12 * want
    assert abs(f.astype("fp32").magnetic(variant=7) - want) < 1e-6 * want


@pytest.mark.parametrize("dims", DIMS[:2])
def test_adjoint_uneven_extents(FL, dims):
    print(f"[tiles] adjoint {dims}", flush=True)
    U = O.random_field(dims, 8200 + dims[1], 0.3)
    Go = O.b2_grad(U)
    scale = np.abs(Go).max()
    f = FL.GaugeField.from_complex(U)
    for g, tol in ((f, 1e-12), (f.astype("fp32"), 1e-5)):
        for v in (0, 1, 2):
            assert np.abs(g.magnetic_grad(variant=v).to_complex().cpu().numpy() - Go).max() < tol * scale, v


@pytest.mark.parametrize("mu", [1, 2, 3])
@pytest.mark.parametrize("kind", ["scaled", "sheared"])
@pytest.mark.parametrize("dims", [(3, 16, 16, 32), (11, 20, 21, 23)])
def test_magnetic_of_links_that_are_not_unitary(FL, dims, kind, mu):
    # FP64 makes no assumption on the links: one link of one direction that is not unitary, in the last
    # tile, and B is that of the quadrant form.  (Both forms add the same leaves: 1e-12.)
    f = FL.GaugeField.random(dims, 5, 0.3, "fp64")
    U = f.to_complex()
    if kind == "scaled":
        U[-1, -1, -1, -1, mu] *= 1.5
    else:
        U[-1, -1, -1, -1, mu, 0] += 0.5 * U[-1, -1, -1, -1, mu, 1]
    g = FL.GaugeField.from_complex(U)
    ref = g.magnetic(variant=1)
    assert abs(ref - f.magnetic(variant=1)) > 1e-9 * ref
    for v in (0, 7):
        assert abs(g.magnetic(variant=v) - ref) < 1e-12 * ref
    assert abs(f.magnetic() - f.magnetic(variant=1)) < 1e-12 * ref   # (the workspace again, clean links)


@pytest.mark.parametrize("mu", [1, 2, 3])
def test_ensemble_of_links_that_are_not_unitary(FL, mu):
    from flue_lat_amd.ensemble import Ensemble
    dims = [(4, 16, 16, 32), (11, 17, 13, 21), (5, 20, 20, 20)]
    e = Ensemble.random(dims, [1, 2, 3], 0.3, "fp64")
    U = e.field(1).to_complex()
    U[-1, -1, -1, -1, mu] *= 1.5
    e.field(1).data.copy_(FL.GaugeField.from_complex(U).data)
    ref = [e.field(c).magnetic(variant=1) for c in range(3)]
    _, B = e.flow(0.01, 0, measure_every=1)
    for c in range(3):
        assert abs(B[0, c] - ref[c]) < 1e-12 * ref[c]


def quadrant_f(f, mu, nu):
    """F by quadrants: the form without a workspace."""
    from flue_lat_amd import _lib
    out = torch.empty((3, 3) + tuple(reversed(f.dims)), dtype=torch.complex128, device=f.device)
    out = out.permute(5, 4, 3, 2, 1, 0)
    st = (ctypes.c_int64 * 6)(*out.stride())
    assert _lib.lib().flue_fmunu(f._cdims, ctypes.c_void_p(f.data.data_ptr()), f.prec, mu, nu, 0,
                                 ctypes.c_void_p(out.data_ptr()), _lib.FLUE_OUT_STRIDED, st,
                                 ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    return out


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-13), ("fp32", 2e-6)])
@pytest.mark.parametrize("dims", [(12, 13, 31, 20), (37, 12, 14, 17), (16, 32, 16, 16)])
def test_fmunu_tiles(FL, dims, prec, tol):
    # every plane in both orientations.  The forms add the same 28 leaves of at most 12 links, of size
    # O(1) each with weights of sum 2.2 or so: FP64 100 eps of the largest entry; FP32 30 eps.
    f = FL.GaugeField.random(dims, 9, 0.3, prec)
    for mu in range(1, 5):
        for nu in range(1, 5):
            if mu == nu:
                continue
            want, got = quadrant_f(f, mu, nu), f.fmunu(mu, nu)
            scale = want.abs().max()
            assert (got - want).abs().max() < tol * scale, (mu, nu)


@pytest.mark.parametrize("mu,nu,d", [(2, 1, 2), (1, 4, 4), (3, 4, 3), (3, 1, 1), (2, 3, 3), (4, 2, 2)])
def test_fmunu_of_links_that_are_not_unitary(FL, mu, nu, d):
    f = FL.GaugeField.random((12, 13, 31, 20), 9, 0.3, "fp64")
    U = f.to_complex()
    U[-1, -1, -1, -1, d - 1] *= 1.5
    g = FL.GaugeField.from_complex(U)
    want = quadrant_f(g, mu, nu)
    assert (quadrant_f(f, mu, nu) - want).abs().max() > 1e-3 * want.abs().max()
    assert torch.equal(g.fmunu(mu, nu), want)


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("dims", [(23, 13, 16, 17), (35, 11, 17, 11), (8, 32, 16, 16), (33, 8, 16, 16), (65, 3, 5, 71)])
def test_fmunu_orders_of_the_output(FL, dims, prec, variant):
    # an output whose t is dense takes the sites of large lattices in another order than one whose x comes
    # before t: the same arithmetic for each site, so the same numbers
    from flue_lat_amd import _lib
    f = FL.GaugeField.random(dims, 21, 0.3, prec)
    for mu in range(1, 5):
        for nu in range(1, 5):
            got = []
            for order in ((5, 4, 3, 2, 1, 0), (0, 1, 2, 3, 4, 5)):
                shape = dims + (3, 3)
                out = torch.full([shape[k] for k in order], float("nan"), dtype=torch.complex128, device=f.device)
                out = out.permute([order.index(k) for k in range(6)])
                st = (ctypes.c_int64 * 6)(*out.stride())
                assert out.shape == shape and _lib.lib().flue_fmunu(
                    f._cdims, ctypes.c_void_p(f.data.data_ptr()), f.prec, mu, nu, variant,
                    ctypes.c_void_p(out.data_ptr()), _lib.FLUE_OUT_STRIDED, st,
                    ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
                got.append(out)
            assert torch.equal(*got), (mu, nu)


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-13), ("fp32", 1e-6)])
@pytest.mark.parametrize("R,T", [(6, 6), (1, 3), (4, 5), (6, 2)])
@pytest.mark.parametrize("dims", [(5, 16, 16, 3), (4, 33, 31, 2), (2, 300, 7, 3), (31, 8, 5, 4), (3, 2, 128, 2)])
def test_wilson_loop_tiles(FL, dims, R, T, prec, tol):
    # planes with x, which take tiles, against the same loops where they do not: with x and the third
    # direction exchanged, and, time in the plane, slice by slice.  Both form the same products (FP64
    # 1e-13; FP32 traces round at 2^-24 of 3, averaged over the sites).
    f = FL.GaugeField.random(dims, 4, 0.3, prec)
    U = f.to_complex()
    for o, s in ((3, 4), (4, 3)):                      # plane (x, o); s the direction outside
        perm = {1: 1, 2: s, s: 2, o: o}                # x and s exchanged
        ax = [perm[d] - 1 for d in (1, 2, 3, 4)]
        V = U.permute(*ax, 4, 5, 6)[..., ax, :, :]
        g = FL.GaugeField.from_complex(V.contiguous(), precision=prec)
        assert np.abs(f.wilson_loops(2, o, R, T) - g.wilson_loops(s, o, R, T)).max() < 3 * tol
        assert np.abs(f.wilson_loops(o, 2, R, T) - g.wilson_loops(o, s, R, T)).max() < 3 * tol
        assert np.abs(f.wilson_loops_slices(2, o, R, T) - g.wilson_loops_slices(s, o, R, T)).max() < 3 * tol
        assert np.abs(f.wilson_loops(2, o, R, T, tau=2) - g.wilson_loops(s, o, R, T, tau=2)).max() < 3 * tol
    for mu, nu in ((1, 2), (2, 1)):
        table = f.wilson_loops(mu, nu, R, T)
        assert np.abs(table - f.wilson_loops_slices(mu, nu, R, T).mean(axis=2)).max() < 3 * tol
