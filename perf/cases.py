"""Performance cases of flue_lat_amd: the work a lattice program has it do, through the
package's public entry points.

A case is a dict of plain values: "op" (below), the extents nt, nx, ny, nz, the link
precision "prec", and the options of the op.  The sizes are those of the package's own
benchmark (48^3x96, ensembles of 16^3 x Nt), of its tests (8^3x16, 16^3x32, 24^3x48) and
generic ragged ones.

ops
  measure   the observables of one resident configuration: three plaquette averages, the
            Polyakov loop and the magnetic B (what a measurement run does per configuration)
  fields    the 5-loop field strength F of all six planes, per site
  loops     the Wilson-loop tables of one temporal and one spatial plane
  flow      Wilson flow of a copy of the field
  force     a differentiated Wilson action: value and link gradient (torch.autograd)
  b2force   a differentiated magnetic B: value and link gradient (torch.autograd)
  b2grad    the Lie gradients of B and of the Wilson action of a resident field
  ensemble  Wilson flow of an ensemble of configurations with periodic measurements
  dropin    observables of a host array through the reference-named functions
"""
import itertools
import math

import numpy as np
import torch

import flue_lat_amd as FL
from flue_lat_amd import autograd
from flue_lat_amd.ensemble import Ensemble
from flue_lat_amd.gluonCalc import wloops

EPS = 0.3        # link disorder of the synthetic fields (as in the benchmark)
FLOW_DT = 0.01   # flow step (as in the benchmark)
BETA = 6.0


def _case(name, op, nt, nx, ny, nz, prec="fp64", **opts):
    return dict(name=name, op=op, nt=nt, nx=nx, ny=ny, nz=nz, prec=prec, **opts)


def listed():
    return [
        # a test-sized configuration: launches and host time decide
        _case("measure-8x16-fp64", "measure", 16, 8, 8, 8),
        # an ordinary configuration in the drop-in precision, extents no multiple of 16
        _case("measure-24x48-fp64", "measure", 48, 24, 24, 24),
        # the benchmark configuration with FP32 links: the largest resident measurement
        _case("measure-48x96-fp32", "measure", 96, 48, 48, 48, "fp32"),
        # field strengths of all planes, as for a topological charge or an action density
        _case("fields-24x48-fp64", "fields", 48, 24, 24, 24, clover=False),
        # static-potential tables of a production-sized lattice
        _case("loops-32x64-fp64", "loops", 64, 32, 32, 32, rmax=6, tmax=6),
        # smoothing a small uneven configuration over many steps
        _case("flow-18x15x20x30-fp64", "flow", 30, 18, 15, 20, steps=10),
        # smoothing the benchmark configuration: an odd number of steps, FP32 links
        _case("flow-48x96-fp32", "flow", 96, 48, 48, 48, "fp32", steps=3),
        # a molecular-dynamics force of a ragged field held as a C-ordered torch tensor
        _case("force-20x22x18x26-fp64", "force", 26, 20, 22, 18, order="C"),
        # forward and backward of B on an ordinary configuration
        _case("b2force-24x48-fp64", "b2force", 48, 24, 24, 24, order="F"),
        # gradients of the benchmark configuration, links and gradients resident
        _case("b2grad-48x96-fp32", "b2grad", 96, 48, 48, 48, "fp32"),
        # many configurations with uneven time extents flowed and measured together
        _case("ensemble-16x16-fp32", "ensemble", 0, 16, 16, 16, "fp32", steps=6, every=3,
              nts="16,24,32,48,64,128,16,24,32,48,64,128,16,32,48,24"),
        # the reference's calling convention: a host array in, numbers out
        _case("dropin-16x32-fp64", "dropin", 32, 16, 16, 16),
    ]


# most sites a drawn case of each op has: those of its largest listed case
_RANGES = {   # op: (smallest extent, largest spatial extent, largest site count, precisions)
    "measure": (8, 48, 48 ** 3 * 96, ("fp64", "fp32")),
    "fields": (8, 24, 24 ** 3 * 48, ("fp64", "fp32")),
    "loops": (8, 32, 32 ** 3 * 64, ("fp64", "fp32")),
    "flow": (8, 48, 48 ** 3 * 96, ("fp64", "fp32")),
    "force": (6, 22, 20 * 22 * 18 * 26, ("fp64", "fp32")),
    "b2force": (6, 24, 24 ** 3 * 48, ("fp64", "fp32")),
    "b2grad": (8, 48, 48 ** 3 * 96, ("fp64", "fp32")),
    "ensemble": (8, 16, 16 ** 3 * 644, ("fp64", "fp32")),
    "dropin": (6, 16, 16 ** 3 * 32, ("fp64",)),
}


def draw(rng):
    op = rng.choice(sorted(_RANGES))
    lo, hi, cap, precs = _RANGES[op]
    prec = rng.choice(precs)
    if op == "flow" or op == "b2grad":
        cap = cap if prec == "fp32" else cap // 2   # an FP64 site costs about twice an FP32 one

    def extent(top):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(top)))))

    while True:
        nx = extent(hi)
        if rng.random() < 0.5:
            ny, nz = nx, nx
        else:   # uneven, odd extents among them
            ny, nz = (max(lo, nx + rng.randint(-4, 4)) for _ in range(2))
        nt = extent(2 * hi)
        if op == "ensemble":
            nts = [extent(128) for _ in range(rng.randint(2, 16))]
            nt = 0
            sites = nx * ny * nz * sum(nts)
        else:
            sites = nx * ny * nz * nt
        if sites <= cap and max(nx, ny, nz) <= hi:
            break
    c = dict(op=op, nt=nt, nx=nx, ny=ny, nz=nz, prec=prec)
    if op == "fields":
        c["clover"] = rng.random() < 0.25
    elif op == "loops":
        c["rmax"], c["tmax"] = rng.randint(2, 6), rng.randint(2, 6)
    elif op == "flow":
        c["steps"] = rng.randint(1, 3)
    elif op in ("force", "b2force"):
        c["order"] = rng.choice("CF")
    elif op == "ensemble":
        c["steps"], c["every"] = rng.randint(2, 6), rng.randint(1, 3)
        c["nts"] = ",".join(str(n) for n in nts)
    return c


# ---------------------------------------------------------------- inputs
#
# Link planes are complex tensors W of shape (4, 3, 3, NT, NZ, NY, NX): W[mu, a, b] is the
# (a, b) element of U_mu on the lattice, mu = 0 time.

def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _mm(A, B):
    """Products of 3x3 matrices held as planes (3, 3, ...)."""
    C = A[:, 0, None] * B[None, 0]
    for k in (1, 2):
        C += A[:, k, None] * B[None, k]
    return C


def _dag(A):
    return A.transpose(0, 1).conj()


def _su3(X):
    """Gram-Schmidt on rows 0 and 1, row 2 their conjugated cross product."""
    def dot(u, v):
        return sum(u[k].conj() * v[k] for k in range(3))
    r0 = X[0] / dot(X[0], X[0]).real.sqrt()
    r1 = X[1] - r0 * dot(r0, X[1])
    r1 = r1 / dot(r1, r1).real.sqrt()
    r2 = torch.stack([r0[1] * r1[2] - r0[2] * r1[1], r0[2] * r1[0] - r0[0] * r1[2],
                      r0[0] * r1[1] - r0[1] * r1[0]]).conj()
    return torch.stack([r0, r1, r2])


def _links(dims, seed):
    """SU(3) links at disorder EPS, independent per link, from the seed alone."""
    nt, nx, ny, nz = dims
    gen = torch.Generator(device=_dev())
    gen.manual_seed(int(seed))
    shape = (nt, nz, ny, nx)
    W = torch.empty((4, 3, 3) + shape, dtype=torch.complex128, device=_dev())
    for mu in range(4):
        c = torch.randn((8,) + shape, dtype=torch.float64, device=_dev(), generator=gen) * (0.5 * EPS)
        X = torch.zeros((3, 3) + shape, dtype=torch.complex128, device=_dev())
        d8 = c[7] / math.sqrt(3.0)
        X[0, 0], X[1, 1], X[2, 2] = 1j * (c[2] + d8), 1j * (d8 - c[2]), -2j * d8
        for (a, b), (p, q) in (((0, 1), (0, 1)), ((0, 2), (3, 4)), ((1, 2), (5, 6))):
            X[a, b] = torch.complex(c[q], c[p])
            X[b, a] = torch.complex(-c[q], c[p])
        E = X + 0.5 * _mm(X, X)
        for a in range(3):
            E[a, a] += 1.0
        W[mu] = _su3(E)
    return W


def _reference_layout(W, order="F"):
    """The (NT, NX, NY, NZ, 4, 3, 3) tensor of link planes, in C or Fortran order."""
    U = W.permute(3, 6, 5, 4, 0, 1, 2)
    if order == "C":
        return U.contiguous()
    return U.permute(6, 5, 4, 3, 2, 1, 0).contiguous().permute(6, 5, 4, 3, 2, 1, 0)


def _dims(case):
    return case["nt"], case["nx"], case["ny"], case["nz"]


def _ens_dims(case):
    return [(int(n), case["nx"], case["ny"], case["nz"]) for n in case["nts"].split(",")]


def _rounded(W, prec):
    return W.to(torch.complex64).to(torch.complex128) if prec == "fp32" else W


def _field(W, prec):
    return FL.GaugeField.from_complex(W.permute(3, 6, 5, 4, 0, 1, 2), prec)


def prepare(case, seed):
    op, prec = case["op"], case["prec"]
    if op == "ensemble":
        e = Ensemble(_ens_dims(case), prec)
        for c, d in enumerate(e.dims):
            e.field(c).data.copy_(_field(_links(d, 1000 * seed + c), prec).data)
        return {"case": case, "ensemble": e, "start": e.data.clone()}
    W = _links(_dims(case), seed)
    if op in ("force", "b2force"):
        return {"case": case, "U": _reference_layout(W, case["order"]).requires_grad_(True)}
    if op == "dropin":
        # what the file readers and f2py programs hold: Fortran-ordered host memory
        return {"case": case, "U": np.asfortranarray(_reference_layout(W).cpu().numpy())}
    return {"case": case, "field": _field(W, prec)}


# planes whose Wilson loops a case tabulates: (x, t) and (x, y)
_LOOP_PLANES = ((2, 1), (2, 3))
_PLANES = tuple(itertools.combinations((1, 2, 3, 4), 2))


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "measure":
        f = state["field"]
        return {"plaq": f.plaquette(1, 4, 4, sync=False)[0], "splaq": f.plaquette(2, 4, 4, sync=False)[0],
                "tplaq": f.plaquette(1, 1, 4, sync=False)[0], "polyakov": f.polyakov(sync=False)[0],
                "B": f.magnetic(sync=False)}
    if op == "fields":
        return [state["field"].fmunu(mu, nu, clover=case["clover"]) for mu, nu in _PLANES]
    if op == "loops":
        return [state["field"].wilson_loops(mu, nu, case["rmax"], case["tmax"]) for mu, nu in _LOOP_PLANES]
    if op == "flow":
        return state["field"].clone().wilson_flow(FLOW_DT, case["steps"]).data
    if op in ("force", "b2force"):
        U = state["U"]
        val = autograd.wilson_action(U, BETA, case["prec"]) if op == "force" else autograd.magnetic(U, case["prec"])
        (grad,) = torch.autograd.grad(val, U)
        return {"value": val.detach(), "grad": grad}
    if op == "b2grad":
        f = state["field"]
        return {"b2": f.magnetic_grad().data, "action": f.wilson_grad(BETA).data}
    if op == "ensemble":
        e = state["ensemble"]
        e.data.copy_(state["start"])
        plaq, B = e.flow(FLOW_DT, case["steps"], measure_every=case["every"])
        return {"plaq": plaq, "B": B, "fields": e.data}
    U = state["U"]
    return {"plaq": wloops.plaquette(U, 1, 4, 4)[0], "polyakov": wloops.polyakov(U)[0], "B": wloops.magnetic(U)}


# ---------------------------------------------------------------- work
#
# Per site, with one 3x3 complex product as 198 flop.  B: per plane 20 chain products, 14
# anti-Hermitian closings (180 flop) and 6 conjugations (300 flop).  Flow stage: 18 products
# for the plaquettes, 24 for the links' forces, 4 for the update.

_B_FLOP = 3 * (20 * 198 + 14 * 180 + 6 * 300)
_PLAQ_FLOP = 6 * (2 * 198 + 36)
_STAGE_FLOP = 46 * 198


def work(case):
    op = case["op"]
    r = 4 if case["prec"] == "fp32" else 8
    if op == "ensemble":
        V = sum(n * x * y * z for n, x, y, z in _ens_dims(case))
        meas = case["steps"] // case["every"] + 1
        return {"bytes": 2 * 72 * r * V, "flops": V * (3 * case["steps"] * _STAGE_FLOP + meas * (_B_FLOP + _PLAQ_FLOP))}
    nt, nx, ny, nz = _dims(case)
    V = nt * nx * ny * nz
    field = 72 * r * V
    if op == "measure":
        return {"bytes": field, "flops": V * (_B_FLOP + 2 * _PLAQ_FLOP + 198)}
    if op == "fields":
        per = 2 * 4 * 198 if case["clover"] else _B_FLOP // 3
        return {"bytes": field + 6 * 144 * V, "flops": V * 6 * per}
    if op == "loops":
        n = case["rmax"] * case["tmax"]
        return {"bytes": field, "flops": 2 * V * (198 * (2 * n + 2 * (case["rmax"] + case["tmax"])) // 2 + 36 * n)}
    if op == "flow":
        return {"bytes": 2 * field, "flops": V * 3 * case["steps"] * _STAGE_FLOP}
    if op == "force":
        return {"bytes": 2 * 576 * V, "flops": V * (_PLAQ_FLOP + 42 * 198 + 4 * 198)}
    if op == "b2force":
        return {"bytes": 2 * 576 * V, "flops": V * (3 * _B_FLOP + 4 * 198)}
    if op == "b2grad":
        return {"bytes": 3 * field, "flops": V * (3 * _B_FLOP + 42 * 198)}
    return {"bytes": 576 * V, "flops": V * (_B_FLOP + _PLAQ_FLOP + 198)}


# ---------------------------------------------------------------- values in 64 bits

_AXIS = {0: -4, 1: -1, 2: -2, 3: -3}   # lattice axis of direction mu in the planes


def _at(A, mu, k):
    """A(x + k mu) for every x."""
    return torch.roll(A, -k, _AXIS[mu]) if k else A


def _retr(A, B):
    """Re Tr(A B^+) per site."""
    return (A * B.conj()).real.sum((0, 1))


def _plaquette_sum(W, mu0, mu1, nu1):
    s = 0.0
    for mu in range(mu0, mu1 + 1):
        for nu in range(mu + 1, nu1 + 1):
            s += _retr(_mm(W[mu], _at(W[nu], mu, 1)), _mm(W[nu], _at(W[mu], nu, 1))).sum().item()
    return s


def _polyakov_sum(W):
    P = W[0][:, :, 0]
    for t in range(1, W.shape[3]):
        P = _mm(P, W[0][:, :, t])
    return (P[0, 0] + P[1, 1] + P[2, 2]).real.sum().item()


_K5 = 1.0 / 180.0
_WEIGHTS = {(1, 1): 19.0 / 9.0 - 55.0 * _K5, (2, 2): 1.0 / 36.0 - 16.0 * _K5, (3, 3): _K5,
            (1, 2): 32.0 * _K5 - 16.0 / 45.0, (2, 1): 32.0 * _K5 - 16.0 / 45.0,
            (1, 3): 1.0 / 30.0 - 3.0 * _K5, (3, 1): 1.0 / 30.0 - 3.0 * _K5}


def _lines(Wm, mu):
    """{n: product of n links along +mu from x} for n = 1..3."""
    L = {1: Wm}
    for n in (2, 3):
        L[n] = _mm(L[n - 1], _at(Wm, mu, n - 1))
    return L


def _leaf_sum(W, mu, nu, shapes):
    """Weighted sum of the loops at x over the four quadrants of (mu, nu), each read
    counter-clockwise from x: for a rectangle with corners x, the four leaves are the one
    loop from its lower-left corner, moved to each corner."""
    Lm, Ln = _lines(W[mu], mu), _lines(W[nu], nu)
    Q = 0.0
    for (a, b), k in shapes.items():
        ca = _mm(Lm[a], _at(Ln[b], mu, a))        # x -> x + a mu -> x + a mu + b nu
        cb = _mm(Ln[b], _at(Lm[a], nu, b))        # x -> x + b nu -> x + a mu + b nu
        loop = _mm(ca, _dag(cb))
        Q = Q + k * loop
        Q = Q + k * _at(_mm(_mm(_dag(Lm[a]), loop), Lm[a]), mu, -a)
        Q = Q + k * _at(_mm(_mm(_dag(Ln[b]), loop), Ln[b]), nu, -b)
        Q = Q + k * _at(_at(_mm(_dag(cb), ca), mu, -a), nu, -b)
    return Q


def _fmunu(W, mu, nu, clover):
    Q = _leaf_sum(W, mu, nu, {(1, 1): 1.0} if clover else _WEIGHTS)
    return ((Q - _dag(Q)) / 8.0).transpose(0, 1)


def _b_density(Ws):
    """Sum over sites of -ReTr F^2 over the spatial planes, for whole time slices Ws."""
    s = 0.0
    for mu, nu in ((2, 1), (1, 3), (3, 2)):
        F = _fmunu(Ws, mu, nu, False)
        s = s + (F.real ** 2 + F.imag ** 2).sum()   # F is anti-Hermitian
    return s


def _slabs(W):
    """Slabs of whole time slices, small enough for the products above."""
    nt, per = W.shape[3], W.shape[4] * W.shape[5] * W.shape[6]
    n = max(1, min(nt, 1500000 // per))
    return [slice(t, min(t + n, nt)) for t in range(0, nt, n)]


def _magnetic(W):
    V = W[0, 0, 0].numel()
    return sum(_b_density(W[:, :, :, sl]).item() for sl in _slabs(W)) / V


def _pta(M):
    T = 0.5 * (M - _dag(M))
    tr = (T[0, 0] + T[1, 1] + T[2, 2]) / 3.0
    T = T.clone()
    for a in range(3):
        T[a, a] -= tr
    return T


def _action_grad(W, mu):
    """P_TA(U_mu Sigma), Sigma the sum of the six staples."""
    S = 0.0
    for nu in range(4):
        if nu == mu:
            continue
        S = S + _mm(_mm(_at(W[nu], mu, 1), _dag(_at(W[mu], nu, 1))), _dag(W[nu]))
        low = _mm(_mm(_dag(_at(W[nu], mu, 1)), _dag(W[mu])), W[nu])
        S = S + _at(low, nu, -1)
    return _pta(_mm(W[mu], S))


def _b2_grad(W):
    """The Lie gradient of B per link: 2 G = P_TA(E U^+) for torch's gradient E."""
    V = W[0, 0, 0].numel()
    G = torch.zeros_like(W)
    for sl in _slabs(W):
        with torch.enable_grad():
            Ws = W[:, :, :, sl].clone().requires_grad_(True)
            (E,) = torch.autograd.grad(_b_density(Ws) / V, Ws)
        for mu in (1, 2, 3):
            G[mu, :, :, sl] = 0.5 * _pta(_mm(E[mu], _dag(Ws.detach()[mu])))
        del E, Ws
    return G


def _expm(X):
    E = X.clone()
    term = X
    for k in range(2, 13):   # |X| is of the order of the flow step
        term = _mm(term, X) / k
        E += term
    for a in range(3):
        E[a, a] += 1.0
    return E


def _flow(W, steps):
    for _ in range(steps):
        acc = torch.zeros_like(W)
        for ca, cb in ((0.0, 0.25), (-17.0 / 9.0, 8.0 / 9.0), (-1.0, 0.75)):
            new = torch.empty_like(W)
            for mu in range(4):
                acc[mu] = ca * acc[mu] - (cb * FLOW_DT) * _action_grad(W, mu)
                new[mu] = _mm(_expm(acc[mu]), W[mu])
            W = new
        for mu in range(4):
            W[mu] = _su3(W[mu])
    return W


def _soa(W):
    """The package's resident layout of link planes: one flat real array."""
    return torch.view_as_real(W.contiguous()).reshape(-1)


def _loop_tables(W, mu, nu, rmax, tmax):
    out = np.empty((rmax, tmax))
    V = W[0, 0, 0].numel()

    def lines(d, n):
        L = [None, W[d]]
        for k in range(1, n):
            L.append(_mm(L[-1], _at(W[d], d, k)))
        return L
    Lm, Ln = lines(mu, rmax), lines(nu, tmax)
    for r in range(1, rmax + 1):
        for t in range(1, tmax + 1):
            ca, cb = _mm(Lm[r], _at(Ln[t], mu, r)), _mm(Ln[t], _at(Lm[r], nu, t))
            out[r - 1, t - 1] = _retr(ca, cb).sum().item() / V
    return out


def _link_grad(G, W):
    """torch's gradient 2 G U in the (NT, NX, NY, NZ, 4, 3, 3) index order."""
    E = torch.stack([2.0 * _mm(G[mu], W[mu]) for mu in range(4)])
    return E.permute(3, 6, 5, 4, 0, 1, 2)


@torch.no_grad()
def exact(case, seed):
    op, prec = case["op"], case["prec"]
    if op == "ensemble":
        dims = _ens_dims(case)
        marks = range(0, case["steps"] + 1, case["every"])
        plaq, B = np.empty((len(marks), len(dims))), np.empty((len(marks), len(dims)))
        fields = []
        for c, d in enumerate(dims):
            W = _rounded(_links(d, 1000 * seed + c), prec)
            done = 0
            for m, k in enumerate(marks):
                W = _flow(W, k - done)
                done = k
                plaq[m, c], B[m, c] = _plaquette_sum(W, 0, 3, 3), _magnetic(W)
            fields.append(_soa(_flow(W, case["steps"] - done)))
        return {"plaq": plaq, "B": B, "fields": torch.cat(fields)}
    W0 = _links(_dims(case), seed)
    W = _rounded(W0, prec)
    V = W[0, 0, 0].numel()
    if op == "measure":
        one = lambda v: torch.tensor([v], dtype=torch.float64)
        return {"plaq": one(_plaquette_sum(W, 0, 3, 3)), "splaq": one(_plaquette_sum(W, 1, 3, 3)),
                "tplaq": one(_plaquette_sum(W, 0, 0, 3)), "polyakov": one(_polyakov_sum(W)), "B": one(_magnetic(W))}
    if op == "fields":
        return [_fmunu(W, mu - 1, nu - 1, case["clover"]).permute(2, 5, 4, 3, 0, 1) for mu, nu in _PLANES]
    if op == "loops":
        return [_loop_tables(W, mu - 1, nu - 1, case["rmax"], case["tmax"]) for mu, nu in _LOOP_PLANES]
    if op == "flow":
        return _soa(_flow(W, case["steps"]))
    if op == "force":
        G = torch.stack([(BETA / 6.0) * _action_grad(W, mu) for mu in range(4)])
        S = BETA * (6.0 * V - _plaquette_sum(W, 0, 3, 3) / 3.0)
        return {"value": torch.tensor(S, dtype=torch.float64), "grad": _link_grad(G, W0)}
    if op == "b2force":
        return {"value": torch.tensor(_magnetic(W), dtype=torch.float64), "grad": _link_grad(_b2_grad(W), W0)}
    if op == "b2grad":
        G = torch.stack([(BETA / 6.0) * _action_grad(W, mu) for mu in range(4)])
        return {"b2": _soa(_b2_grad(W)), "action": _soa(G)}
    return {"plaq": _plaquette_sum(W, 0, 3, 3), "polyakov": _polyakov_sum(W), "B": _magnetic(W)}
