"""The Wilson flow of plain FP64 links that are not SU(3): nothing is assumed about the links of such a
field, so on every lattice size it is the flow by staple sums of whole links (flue_flow_stage).

Each stage's rounding is some 1e-15 of links of size one, for both stencils and each of at most three
steps; 1e-12 is far above that and far below what one spoiled link changes.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

EPS = 0.02
# below and above the 32,768 sites from which untuned flows take the plaquette-first stencil, the last in boxes
DIMS = [(7, 11, 12, 13), (23, 11, 12, 13), (2, 33, 34, 31)]


@pytest.fixture(scope="module")
def FL():
    import flue_lat_amd as FL
    return FL


def spoil(U, kind):
    """One link of the last time slice, spoiled so that rows 0 and 1 do not give row 2."""
    link = U[-1, 3, 2, 5, 2]
    if kind == "scaled":
        link *= 1.5
    elif kind == "phase":
        link *= np.exp(0.4j)
    elif kind == "row 2":
        link[2] += 0.5 * link[0]
    elif kind == "tiny":
        link[2] *= 1.0 + 1e-6
    else:
        link[2, 1] = complex("nan")


def by_stages(FL, g, nsteps):
    """The flow of a copy of g from the single-stage entry, which takes staple sums."""
    from flue_lat_amd import _lib
    a, b = g.data.clone(), torch.empty_like(g.data)
    acc = torch.empty(32 * g.V, dtype=torch.float64, device=g.device)
    for k in range(3 * nsteps):
        _lib.check(_lib.lib().flue_flow_stage(g._cdims, ctypes.c_void_p(a.data_ptr()), g.prec,
                                              ctypes.c_void_p(b.data_ptr()), ctypes.c_void_p(acc.data_ptr()), EPS,
                                              k % 3, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)),
                   "flue_flow_stage")
        a, b = b, a
    return a


def assert_same(got, want):
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(got), nan)
    assert float(torch.where(nan, 0.0, got - want).abs().max()) < 1e-12


@pytest.mark.parametrize("kind", ["scaled", "phase", "row 2", "tiny", "nan"])
@pytest.mark.parametrize("dims", DIMS)
def test_flow_of_links_that_are_not_su3(FL, dims, kind):
    f = FL.GaugeField.random(dims, 77, 0.3, "fp64")
    U = f.to_complex()
    spoil(U, kind)
    g = FL.GaugeField.from_complex(U)
    # an odd last step alone, a pair alone, pairs with an odd step, as a graph and without
    for nsteps, use_graph in ((1, False), (2, True), (3, False), (4, True), (5, True)):
        W = g.clone()
        W.wilson_flow(EPS, nsteps, use_graph=use_graph)
        assert_same(W.data, by_stages(FL, g, nsteps))
    # clean links afterwards (library buffers hold what the flows left)
    W = f.clone()
    W.wilson_flow(EPS, 2, use_graph=False)
    assert_same(W.data, by_stages(FL, f, 2))


@pytest.mark.parametrize("kind", ["scaled", "phase", "row 2", "nan"])
def test_ensemble_flow_of_links_that_are_not_su3(FL, kind):
    # two of four configurations spoiled, the second of them the smallest; the others are not affected
    from flue_lat_amd.ensemble import Ensemble
    dims = [(9, 11, 12, 13), (17, 12, 9, 8), (3, 4, 5, 6), (14, 8, 10, 12)]
    for nsteps, use_graph in ((1, False), (3, True)):
        e = Ensemble.random(dims, [5, 6, 7, 8], 0.3, "fp64")
        clean = e.data.clone()
        e.flow(EPS, nsteps, measure_every=0, use_graph=use_graph)
        flowed = e.data.clone()
        e.data.copy_(clean)
        want = []
        for c in range(4):
            g = e.field(c)
            if c in (1, 2):
                U = g.to_complex()
                spoil(U, kind)
                g.data.copy_(FL.GaugeField.from_complex(U).data)
            want.append(by_stages(FL, g, nsteps))
        e.flow(EPS, nsteps, measure_every=0, use_graph=use_graph)
        for c in range(4):
            assert_same(e.field(c).data, want[c])
        for c in (0, 3):
            lo, hi = int(e.offsets[c]), int(e.offsets[c + 1])
            assert torch.equal(e.data[lo:hi], flowed[lo:hi])
