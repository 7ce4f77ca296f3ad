"""Visit orders and untuned forms of the flow and gradient stencils.

Every order of one stencil runs the same per-link code on the same neighbours, so its fields
are bit-identical; lattices whose rows do not divide the boxes leave partial boxes and
blocks.  The untuned flow (plaquette-first from 32768 sites, in boxes on slices of 32768 sites)
is compared with the staple sums: both are FP64-accurate per stage, and links differ by
rounding of the force times the step, far below 1e-12 (FP64) and 2e-6 (FP32 links: a few
roundings of a unit entry, the bound the flow's other tests use).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def FL():
    import flue_lat_amd as FL
    return FL


def force(FL, tmp_path, dims, prec, variant):
    p = tmp_path / f"tune_{variant}.txt"
    p.write_text(f"0 3 {0 if prec == 'fp64' else 1} {dims[0]} {dims[1]} {dims[2]} {dims[3]} {variant} 1.0\n")
    FL.field.tune_load(p)


def flowed(f, steps=1):
    g = f.clone()
    g.wilson_flow(0.02, steps, use_graph=False)
    return g.data


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("dims", [(3, 40, 7, 11), (2, 50, 23, 5), (5, 3, 65, 17), (1, 7000, 1, 2)])
def test_orders_bit_identical(FL, tmp_path, dims, prec):
    # (1, 7000, 1, 2): no row fits the smaller boxes, so they take the storage order
    print(f"[orders] {dims} {prec}", flush=True)
    f = FL.GaugeField.random(dims, 17, 0.3).astype(prec)
    for group in ((1, 2, 3, 4, 5, 6), (7, 8, 9, 10, 11, 12, 13)):
        want = None
        for v in group:
            force(FL, tmp_path, dims, prec, v)
            got = flowed(f), f.wilson_grad(6.0).data
            if want is None:
                want = got
            assert all(torch.equal(a, b) for a, b in zip(got, want)), v


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 2e-6)])
@pytest.mark.parametrize("dims", [(4, 33, 32, 31), (3, 37, 33, 31), (8, 16, 16, 16), (9, 16, 16, 15)])
def test_untuned_flow_matches_staple_sums(FL, tmp_path, dims, prec, tol):
    # both sides of the two thresholds, and an extent that leaves partial boxes
    print(f"[flow] {dims} {prec}", flush=True)
    f = FL.GaugeField.random(dims, 23, 0.3).astype(prec)
    untuned = flowed(f, 3)
    force(FL, tmp_path, dims, prec, 1)
    assert float((untuned - flowed(f, 3)).abs().max()) < tol


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-13), ("fp32", 1e-6)])
@pytest.mark.parametrize("dims", [(1, 1, 1, 1), (2, 3, 1, 5), (16, 8, 8, 8), (5, 13, 16, 16), (9, 29, 31, 33), (64, 16, 16, 17)])
def test_untuned_plaquette(FL, dims, prec, tol):
    # the untuned forms by size (a thread per site and plane, walks of 2 to 6 slices), for every range
    # of planes, against the loops walked link by link
    f = FL.GaugeField.random(dims, 6, 0.3, prec)
    loop = {(mu, nu): f.wilson_loop(mu, nu, 1, 1) for mu in range(1, 5) for nu in range(mu + 1, 5)}
    V = np.prod(dims)
    for mu0 in range(1, 5):
        for mu1 in range(1, 5):
            for nu1 in range(1, 5):
                want = V * sum(v for (mu, nu), v in loop.items() if mu0 <= mu <= mu1 and nu <= nu1)
                assert abs(f.plaquette(mu0, mu1, nu1)[0] - want) <= tol * 18 * V, (mu0, mu1, nu1)


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-13), ("fp64-su3", 1e-13), ("fp32", 1e-7)])
@pytest.mark.parametrize("dims", [(1, 1, 1, 1), (1, 2, 3, 4), (3, 3, 7, 1), (4, 4, 4, 4), (13, 5, 5, 13), (16, 10, 8, 8),
                                  (4, 16, 16, 16), (5, 16, 16, 16)])
def test_untuned_magnetic_of_small_lattices(FL, dims, prec, tol):
    # a wave per quadrant, partial blocks of 64 sites and the sizes at which other forms take over,
    # against a thread per site.  FP32: the four parts of a site round at 2^-24 once more each.
    f = FL.GaugeField.random(dims, 8, 0.3, "fp64").astype(prec)
    want = f.magnetic(variant=1)
    assert abs(f.magnetic() - want) <= tol * abs(want)
