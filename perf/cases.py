"""The work that users of lmhip have it do, as timed cases.

Each case is one call of a public entry point of the host package: a whole
`Evolution` of a density matrix or of kets over a short timeline, a batch of
disorder realisations, the gradient of an evolution, or a density matrix from
a kept eigensystem.  Sizes and models are those of the benchmark's workloads
and the tests (squares from 10 x 10 to 100 x 100, honeycombs up to 120 x 120
cells, ket evolutions at N ~ 10^5), with odd and ragged ones between them.

A run returns device matrices as torch views of the library's memory.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "latticemodels.jl_amd"))

import lmhip  # noqa: E402

DENSE_P0_MAX = 12000        # above: P0 is a half-filled product state, given by its entries
T2, MASS = 0.1, 0.2         # Haldane model: next-nearest hopping, sublattice mass


def listed():
    return [
        # a small flux-threading run with every observable read at every step: launches and latency
        {"name": "small_flux_10", "kind": "evolve", "lattice": "square", "l1": 10, "l2": 10, "periodic": "none",
         "field": "flux", "strength": 0.2, "disorder": 0.0, "dt": 0.1, "steps": 20, "observe": 1},
        # a narrow disordered cylinder of odd sides in a Landau field, observables now and then
        {"name": "cylinder_37x23", "kind": "evolve", "lattice": "square", "l1": 37, "l2": 23, "periodic": "axis2",
         "field": "landau", "strength": 0.02, "disorder": 2.0, "dt": 0.05, "steps": 20, "observe": 5},
        # the headline workload: a disordered torus, Landau field ramped, N = 10^4
        {"name": "torus_100", "kind": "evolve", "lattice": "square", "l1": 100, "l2": 100, "periodic": "both",
         "field": "landau", "strength": 0.01, "disorder": 1.0, "dt": 0.05, "steps": 10, "observe": 10},
        # flux insertion on a mid-size disordered square: bonds that differ from site to site
        {"name": "flux_48", "kind": "evolve", "lattice": "square", "l1": 48, "l2": 48, "periodic": "none",
         "field": "flux", "strength": 0.2, "disorder": 1.0, "dt": 0.1, "steps": 10, "observe": 10},
        # flux insertion in a Chern insulator (Haldane), N = 3200, nine neighbours per site
        {"name": "haldane_40", "kind": "evolve", "lattice": "honeycomb", "l1": 40, "l2": 40, "periodic": "none",
         "field": "flux", "strength": 0.5, "disorder": 0.0, "dt": 0.02, "steps": 5, "observe": 5},
        # the same at the benchmark's largest size, N = 28800: 13.3 GB per matrix
        {"name": "haldane_120", "kind": "evolve", "lattice": "honeycomb", "l1": 120, "l2": 120, "periodic": "none",
         "field": "flux", "strength": 0.5, "disorder": 0.0, "dt": 0.02, "steps": 2, "observe": 2},
        # an ensemble of disorder realisations of uneven size advanced together
        {"name": "ensemble_12", "kind": "batch", "members": 12, "lmin": 24, "lmax": 64, "strength": 0.005,
         "disorder": 2.0, "dt": 0.05, "steps": 4},
        # one ket at N ~ 10^5 by Krylov, its density read at every step
        {"name": "krylov_224", "kind": "krylov", "l1": 224, "l2": 224, "strength": 3.0 * 1.519e-3, "dt": 0.1,
         "steps": 20, "kets": 1},
        # a block of kets (scattering states) under the Taylor step
        {"name": "ketblock_64", "kind": "kets", "lattice": "square", "l1": 64, "l2": 64, "periodic": "none",
         "field": "flux", "strength": 0.2, "disorder": 1.0, "dt": 0.1, "steps": 20, "kets": 48},
        # the differentiation workload: forward with tape, then gradients of a density loss
        {"name": "gradient_32", "kind": "gradient", "lattice": "square", "l1": 32, "l2": 32, "periodic": "none",
         "field": "flux", "strength": 0.2, "disorder": 0.3, "dt": 0.1, "steps": 10, "every": 5},
        # the same for a Haldane flake too large for the on-chip reverse sweep
        {"name": "gradient_haldane_36", "kind": "gradient", "lattice": "honeycomb", "l1": 36, "l2": 36,
         "periodic": "none", "field": "flux", "strength": 0.5, "disorder": 0.1, "dt": 0.02, "steps": 5, "every": 5},
        # a thermal density matrix from a kept eigensystem (a temperature or mu scan)
        {"name": "thermal_48", "kind": "thermal", "l1": 48, "l2": 48, "strength": 0.01, "disorder": 1.0,
         "temperature": 0.2, "mu": 0.3},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sides(rng, lo, hi):
    """Two sides whose product is spread over lo^2 .. hi^2 on a log scale."""
    side = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    aspect = math.exp(rng.uniform(-0.5, 0.5))
    return (max(lo, min(hi, int(round(side * aspect)))), max(lo, min(hi, int(round(side / aspect)))))


def draw(rng):
    kind = rng.choice(["strip", "strip", "flux", "flux", "haldane", "haldane", "batch", "krylov", "kets", "gradient",
                       "gradient_haldane", "thermal"])
    if kind == "strip":
        l1, l2 = _sides(rng, 10, 100)
        return {"kind": "evolve", "lattice": "square", "l1": l1, "l2": l2,
                "periodic": rng.choice(["none", "axis1", "axis2", "both"]), "field": "landau",
                "strength": rng.uniform(0.002, 0.05), "disorder": rng.choice([0.0, 1.0, 2.0]),
                "dt": rng.choice([0.05, 0.1]), "steps": rng.randint(3, 10), "observe": rng.randint(1, 10)}
    if kind == "flux":
        l1, l2 = _sides(rng, 10, 80)
        return {"kind": "evolve", "lattice": "square", "l1": l1, "l2": l2, "periodic": "none",
                "field": rng.choice(["flux", "symmetric"]), "strength": rng.uniform(0.005, 0.3),
                "disorder": rng.choice([0.0, 1.0]), "dt": rng.choice([0.05, 0.1]), "steps": rng.randint(3, 10),
                "observe": rng.randint(1, 10)}
    if kind == "haldane":
        l1, l2 = _sides(rng, 8, 100)
        return {"kind": "evolve", "lattice": "honeycomb", "l1": l1, "l2": l2, "periodic": "none", "field": "flux",
                "strength": rng.uniform(0.1, 0.5), "disorder": rng.choice([0.0, 0.2]), "dt": 0.02, "steps": 2,
                "observe": 2}
    if kind == "batch":
        lmin = rng.randint(10, 32)
        return {"kind": "batch", "members": rng.randint(3, 12), "lmin": lmin, "lmax": rng.randint(lmin, 64),
                "strength": rng.uniform(0.002, 0.02), "disorder": 2.0, "dt": 0.05, "steps": rng.randint(1, 6)}
    if kind == "krylov":
        l1, l2 = _sides(rng, 20, 224)
        return {"kind": "krylov", "l1": l1, "l2": l2, "strength": rng.uniform(0.001, 0.01), "dt": 0.1,
                "steps": rng.randint(3, 20), "kets": rng.choice([1, 1, 3])}
    if kind == "kets":
        l1, l2 = _sides(rng, 10, 100)
        field = rng.choice(["flux", "landau"])
        return {"kind": "kets", "lattice": "square", "l1": l1, "l2": l2,
                "periodic": "none" if field == "flux" else rng.choice(["none", "both"]), "field": field, "strength": rng.uniform(0.01, 0.2),
                "disorder": rng.choice([0.0, 1.0]), "dt": 0.1, "steps": rng.randint(3, 20), "kets": _log_int(rng, 2, 96)}
    if kind == "gradient":
        l1, l2 = _sides(rng, 8, 32)
        return {"kind": "gradient", "lattice": "square", "l1": l1, "l2": l2, "periodic": "none", "field": "flux",
                "strength": rng.uniform(0.05, 0.3), "disorder": 0.3, "dt": 0.1, "steps": rng.randint(2, 10),
                "every": rng.randint(2, 10)}
    if kind == "gradient_haldane":
        l1, l2 = _sides(rng, 20, 40)
        return {"kind": "gradient", "lattice": "honeycomb", "l1": l1, "l2": l2, "periodic": "none", "field": "flux",
                "strength": rng.uniform(0.1, 0.5), "disorder": 0.1, "dt": 0.02, "steps": rng.randint(2, 5),
                "every": rng.randint(2, 5)}
    l1, l2 = _sides(rng, 8, 48)
    return {"kind": "thermal", "l1": l1, "l2": l2, "strength": rng.uniform(0.005, 0.05), "disorder": 1.0,
            "temperature": rng.uniform(0.05, 0.5), "mu": rng.uniform(-1.0, 1.0)}


# ------------------------------------------------------------ inputs of a case

def _sites(case):
    return case["l1"] * case["l2"] * (2 if _lattice_kind(case) == "honeycomb" else 1)


def _lattice_kind(case):
    return "honeycomb" if case["kind"] == "krylov" else case.get("lattice", "square")


def _periodic(case):
    p = case.get("periodic", "none")
    return (p in ("axis1", "both"), p in ("axis2", "both"))


def _flux_point(case):
    """A point with no site and no bond on it, near the middle of the lattice."""
    if _lattice_kind(case) == "honeycomb":
        c1, c2 = case["l1"] // 2, case["l2"] // 2
        return (c1 + 0.5 * c2 - 0.5, c2 * math.sqrt(3.0) / 2.0 - math.sqrt(3.0) / 6.0)
    return (case["l1"] // 2 + 0.5, case["l2"] // 2 + 0.5)


def _duration(case):
    return case["dt"] * case["steps"]


def _onsite(case, n, rng):
    w = case.get("disorder", 0.0)
    return rng.uniform(-w / 2.0, w / 2.0, n) if w else None


def _strength_factor(rng):
    return float(rng.uniform(0.9, 1.1))


def _orthonormal(n, r, rng):
    q, _ = np.linalg.qr(rng.normal(size=(n, r)) + 1j * rng.normal(size=(n, r)))
    return q


def _initial(n, rng):
    """A rank-r orthogonal projector as its factor Q (P0 = Q Q^H), or the
    occupied sites of a product state."""
    if n <= DENSE_P0_MAX:
        return "factor", _orthonormal(n, max(4, min(64, n // 16)), rng)
    return "sites", np.sort(rng.permutation(n)[: n // 2])


class _Entries:
    """P given by its nonzero entries."""

    def __init__(self, sites):
        self.rows = self.cols = np.asarray(sites, dtype=np.int64)
        self.vals = np.ones(len(self.rows), dtype=np.complex128)


class _Matrix:
    """A device matrix (column-major, leading dimension ld) for torch."""

    def __init__(self, state):
        p, ld = state.device_ptr()
        self.state = state
        self.__cuda_array_interface__ = {"shape": (state.n, state.n), "typestr": "<c16", "data": (p, False),
                                         "strides": (16, 16 * ld), "version": 3}


def _view(state):
    return torch.as_tensor(_Matrix(state), device="cuda")


def _model(case, rng):
    """Lattice, on-site energies and t -> H(t) of a case, from its seed."""
    l1, l2 = case["l1"], case["l2"]
    per = [("axis1", True)] * _periodic(case)[0] + [("axis2", True)] * _periodic(case)[1]
    honey = _lattice_kind(case) == "honeycomb"
    lat = (lmhip.HoneycombLattice if honey else lmhip.SquareLattice)(l1, l2, boundaries=tuple(per))
    V = _onsite(case, len(lat), rng)
    field = _field(case, _strength_factor(rng))
    terms = () if V is None else (V,)
    if honey:
        return lat, V, lambda t: lmhip.haldane(lat, 1.0, T2, MASS, *terms, field=field(t))
    return lat, V, lambda t: lmhip.tightbinding_hamiltonian(lat, *terms, field=field(t))


def _field(case, factor):
    """t -> field, ramped linearly from 30 % to 100 % over the timeline."""
    top, T = case["strength"] * factor, _duration(case)
    a = lambda t: top * (0.3 + 0.7 * t / T)
    name = case["field"]
    if name == "landau":
        return lambda t: lmhip.LandauGauge(a(t))
    if name == "symmetric":
        return lambda t: lmhip.SymmetricGauge(a(t))
    pt = _flux_point(case)
    return lambda t: lmhip.PointFlux(a(t), pt)


def _times(case):
    return [case["dt"] * k for k in range(case["steps"] + 1)]


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    return {"evolve": _prepare_evolve, "batch": _prepare_batch, "krylov": _prepare_krylov, "kets": _prepare_kets,
            "gradient": _prepare_gradient, "thermal": _prepare_thermal}[case["kind"]](case, rng)


def run(state):
    return state["run"](state)


def _prepare_evolve(case, rng):
    lat, V, h = _model(case, rng)
    solver = lmhip.HIPExp(ctx=lmhip.Context(0))
    form, x = _initial(len(lat), rng)
    if form == "factor":
        q = torch.from_numpy(x).cuda()
        p0 = (q @ q.conj().T).cpu().numpy()
        solver.ctx.set_hamiltonian(h(0.0))
        p0 = lmhip.DensityMatrix.from_array(solver.ctx, p0)
    else:
        p0 = _Entries(x)
    return {"run": _run_evolve, "h": h, "solver": solver, "p0": p0, "times": _times(case), "observe": case["observe"]}


def _run_evolve(s):
    ev = lmhip.Evolution(s["solver"], s["h"], s["p0"])
    rhos, currents = [], []
    for k, (P, H, t) in enumerate(ev(s["times"])):
        if k and k % s["observe"] == 0:
            rho, J = lmhip.observables(P, H)
            rhos.append(rho)
            currents.append(J)
    return {"P": _view(ev.states[0]), "rho": np.array(rhos), "J": np.array(currents)}


def _batch_sides(case):
    """The members' sides: the case's own (the disorder and the states are the seed's)."""
    rng = np.random.default_rng(case["members"] * 10007 + case["lmin"] * 101 + case["lmax"])
    return [int(rng.integers(case["lmin"], case["lmax"] + 1)) for _ in range(case["members"])]


def _prepare_batch(case, rng):
    members = []
    for L in _batch_sides(case):
        n = L * L
        V = _onsite(case, n, rng)
        occ = np.sort(rng.permutation(n)[: n // 2])
        H = lmhip.tightbinding_hamiltonian(lmhip.SquareLattice(L, L), V, field=lmhip.LandauGauge(case["strength"]))
        members.append((H, _Entries(occ)))
    return {"run": _run_batch, "batch": lmhip.BatchedEvolution(members, case["dt"]), "steps": case["steps"]}


def _run_batch(s):
    s["batch"].step(s["steps"])
    return {"P": [_view(P) for P in s["batch"].states], "mean_density": s["batch"].mean_density()}


def _krylov_onsite(xy):
    c = 0.5 * (xy.min(axis=0) + xy.max(axis=0))
    rad = 0.5 * float(np.min(xy.max(axis=0) - xy.min(axis=0)))
    return np.where(np.sum((xy - c) ** 2, axis=1) < rad * rad / 4.0, 0.2, 0.0)


def _random_kets(n, m, rng):
    psi = rng.normal(size=(n, m)) + 1j * rng.normal(size=(n, m))
    return psi / np.linalg.norm(psi, axis=0)


def _prepare_krylov(case, rng):
    lat = lmhip.HoneycombLattice(case["l1"], case["l2"])
    V = _krylov_onsite(lat.coords)
    top, T = case["strength"] * _strength_factor(rng), _duration(case)
    h = lambda t: lmhip.tightbinding_hamiltonian(lat, V, t1=-2.8, field=lmhip.SymmetricGauge(top * (0.3 + 0.7 * t / T)))
    psi = _random_kets(len(lat), case["kets"], rng)
    solver = lmhip.HIPKrylovExp(ctx=lmhip.Context(0))
    solver.ctx.set_hamiltonian(h(0.0))
    kets = lmhip.Kets.from_array(solver.ctx, psi[:, 0] if case["kets"] == 1 else psi)
    return {"run": _run_krylov, "h": h, "solver": solver, "kets": kets, "times": _times(case)}


def _run_krylov(s):
    ev = lmhip.Evolution(s["solver"], s["h"], s["kets"])
    rhos = []
    for k, (psi, H, t) in enumerate(ev(s["times"])):
        if k:
            rhos.append(lmhip.localdensity(psi))
    return {"psi": ev.states[0].to_numpy(), "rho": np.array(rhos)}


def _prepare_kets(case, rng):
    lat, V, h = _model(case, rng)
    solver = lmhip.HIPExp(ctx=lmhip.Context(0))
    solver.ctx.set_hamiltonian(h(0.0))
    kets = lmhip.Kets.from_array(solver.ctx, _random_kets(len(lat), case["kets"], rng))
    return {"run": _run_kets, "h": h, "solver": solver, "kets": kets, "times": _times(case)}


def _run_kets(s):
    ev = lmhip.Evolution(s["solver"], s["h"], s["kets"])
    for psi, H, t in ev(s["times"]):
        pass
    rho, J = ev.states[0].observables(0)
    return {"psi": ev.states[0].to_numpy(), "rho": rho, "J": J}


def _loss_sites(case):
    """A quarter of the sites, the first ones: the corner of the lattice."""
    return np.arange(max(1, _sites(case) // 4))


def _prepare_gradient(case, rng):
    lat, V, h = _model(case, rng)
    solver = lmhip.HIPExp(ctx=lmhip.Context(0))
    q = torch.from_numpy(_initial(len(lat), rng)[1]).cuda()
    solver.ctx.set_hamiltonian(h(0.0))
    p0 = lmhip.DensityMatrix.from_array(solver.ctx, (q @ q.conj().T).cpu().numpy())
    sites = _loss_sites(case)
    weights = rng.uniform(0.5, 1.5, len(sites))
    return {"run": _run_gradient, "h": h, "solver": solver, "p0": p0, "times": _times(case), "every": case["every"],
            "cotangent": lmhip.localdensity_cotangent(len(lat), weights, sites=sites)}


def _run_gradient(s):
    ev = lmhip.Evolution(s["solver"], s["h"], s["p0"])
    tape = lmhip.EvolutionTape(ev, s["every"])
    for P, H, t in ev(s["times"]):
        pass
    rho = lmhip.localdensity(ev.states[0])
    g = tape.backward(s["cotangent"])
    tape.close()
    return {"rho": rho, "field": g.field, "onsite": g.onsite, "P0": _view(g.P0)}


def _prepare_thermal(case, rng):
    lat = lmhip.SquareLattice(case["l1"], case["l2"])
    V = _onsite(case, len(lat), rng)
    H = lmhip.tightbinding_hamiltonian(lat, V, field=lmhip.LandauGauge(case["strength"] * _strength_factor(rng)))
    return {"run": _run_thermal, "eig": lmhip.diagonalize(H, ctx=lmhip.Context(0)), "T": case["temperature"],
            "mu": case["mu"]}


def _run_thermal(s):
    return {"P": _view(lmhip.densitymatrix(s["eig"], T=s["T"], mu=s["mu"]))}


# ------------------------------------------------------------- floors of a case

def _slots(case):
    return 9 if _lattice_kind(case) == "honeycomb" and case["kind"] != "krylov" else 3 if case["kind"] == "krylov" else 4


def _terms(case):
    """About the number of Taylor terms of one step (threshold 1e-10)."""
    growth = (4.0 if _slots(case) == 9 else 4.0 + 0.5 * case.get("disorder", 0.0)) * case["dt"]
    k, term = 0, 1.0
    while term > 1e-10:
        k += 1
        term *= growth / k
    return k


def work(case):
    kind = case["kind"]
    z = _slots(case)
    if kind == "batch":
        s2 = float(sum(L ** 4 for L in _batch_sides(case)))
        return {"bytes": 32.0 * s2, "flops": case["steps"] * 2.0 * _terms(case) * s2 * (8 * z + 6)}
    n = float(_sites(case))
    if kind == "evolve":
        return {"bytes": 32.0 * n * n, "flops": case["steps"] * 2.0 * _terms(case) * n * n * (8 * z + 6)}
    if kind == "kets":
        return {"bytes": 32.0 * n * case["kets"],
                "flops": case["steps"] * float(_terms(case)) * n * case["kets"] * (8 * z + 6)}
    if kind == "krylov":
        # about 14 products by H, two inner products and updates each, per step
        return {"bytes": n * (32.0 * case["kets"] + 8.0 * case["steps"]),
                "flops": case["steps"] * 14.0 * n * case["kets"] * (8 * z + 40)}
    if kind == "gradient":
        # forward, the states back, the costate back, and one sweep for the gradient
        return {"bytes": 64.0 * n * n, "flops": case["steps"] * 8.0 * _terms(case) * n * n * (8 * z + 6)}
    # the Hermitian half of V f V^H
    return {"bytes": 32.0 * n * n, "flops": 4.0 * n ** 3}


# ---------------------------------------------- 64-bit values without the library

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _bonds(kind, l1, l2, periodic, nnn):
    """Bond arrays i, j, r_i, unwrapped r_j, amplitude."""
    nb = 2 if kind == "honeycomb" else 1
    a = np.array([[1.0, 0.0], [0.5, math.sqrt(3.0) / 2.0]] if nb == 2 else [[1.0, 0.0], [0.0, 1.0]])
    basis = np.array([[0.0, 0.0], [0.5, math.sqrt(3.0) / 6.0]])[:nb]
    if nb == 2:
        hops = [(0, 1, 0, -1, 1.0), (0, 1, -1, 0, 1.0), (0, 1, 0, 0, 1.0)]
        if nnn:
            hops += [(0, 0, 1, 0, 1j), (1, 1, -1, 0, 1j), (0, 0, 0, -1, 1j), (1, 1, 0, 1, 1j), (0, 0, -1, 1, 1j),
                     (1, 1, 1, -1, 1j)]
    else:
        hops = [(0, 0, 1, 0, 1.0), (0, 0, 0, 1, 1.0)]
    j1, j2 = (x.ravel() for x in np.meshgrid(np.arange(l1), np.arange(l2), indexing="ij"))
    pos = lambda u, v, b: (u + 1.0)[:, None] * a[0] + (v + 1.0)[:, None] * a[1] + basis[b]
    out = []
    for b0, b1, d1, d2, amp in hops:
        u, v = j1 + d1, j2 + d2
        ok = np.ones(len(u), dtype=bool)
        if not periodic[0]:
            ok &= (u >= 0) & (u < l1)
        if not periodic[1]:
            ok &= (v >= 0) & (v < l2)
        i = (j1 * l2 + j2) * nb + b0
        j = ((u % l1) * l2 + v % l2) * nb + b1
        out.append((i[ok], j[ok], pos(j1, j2, b0)[ok], pos(u, v, b1)[ok], np.full(int(ok.sum()), amp, dtype=complex)))
    return [np.concatenate(x) for x in zip(*out)]


def _unit_integrals(name, pt, ri, rj):
    """Line integral of the vector potential along each bond at strength 1."""
    x1, y1, x2, y2 = ri[:, 0], ri[:, 1], rj[:, 0], rj[:, 1]
    if name == "landau":
        return (x1 + x2) * (y2 - y1) / 2.0
    if name == "symmetric":
        return (x1 * y2 - x2 * y1) / 2.0
    ax, ay, bx, by = x1 - pt[0], y1 - pt[1], x2 - pt[0], y2 - pt[1]
    cosang = (ax * bx + ay * by) / (np.sqrt(ax * ax + ay * ay) * np.sqrt(bx * bx + by * by)) / (1.0 + 1e-11)
    return np.arccos(cosang) * np.sign(ax * by - bx * ay) / (2.0 * math.pi)


class _Exact:
    """H(t) of a case as gathered rows, on torch in complex128."""

    def __init__(self, kind, l1, l2, periodic, field, pt, V, hop, nnn):
        i, j, ri, rj, amp = _bonds(kind, l1, l2, periodic, nnn)
        self.n = l1 * l2 * (2 if kind == "honeycomb" else 1)
        amp = np.where(amp.imag != 0, T2 * amp, hop * amp)
        g = _unit_integrals(field, pt, ri, rj)
        d = np.zeros(self.n) if V is None else np.array(V, dtype=float)
        if nnn:
            d += np.where(np.arange(self.n) % 2 == 0, MASS, -MASS)
        dev = _device()
        rows = np.concatenate([i, j])
        order = np.argsort(rows, kind="stable")
        slot = np.arange(len(rows)) - np.searchsorted(rows[order], rows[order])
        z = int(slot.max()) + 1
        idx, src = np.zeros((z, self.n), dtype=np.int64), np.full((z, self.n), -1, dtype=np.int64)
        idx[slot, rows[order]] = np.concatenate([j, i])[order]
        src[slot, rows[order]] = order
        put = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(dev)
        self.i, self.j, self.amp, self.g, self.d = put(i), put(j), put(amp), put(g), put(d)
        self.idx, self.src = put(idx), put(src)

    def bond_values(self, a):
        return self.amp * torch.exp(-2j * math.pi * (a * self.g))

    def rows(self, a):
        v = self.bond_values(a)
        both = torch.cat([v, v.conj().resolve_conj(), torch.zeros(1, dtype=v.dtype, device=v.device)])
        return both[self.src]           # src -1: the zero at the end

    def dense(self, a, d=None):
        v = self.bond_values(a)
        H = torch.zeros((self.n, self.n), dtype=torch.complex128, device=v.device)
        H = H.index_put((self.i, self.j), v, accumulate=True)
        H = H.index_put((self.j, self.i), v.conj(), accumulate=True)
        return H + torch.diag((self.d if d is None else d).to(torch.complex128))

    def propagate(self, a, dt, X):
        """exp(-i dt H) X, in blocks of columns."""
        v = self.rows(a)
        step = max(1, int(2e9 // (16 * self.n)))
        out = torch.empty_like(X)
        for c in range(0, X.shape[1], step):
            t = X[:, c:c + step].clone()
            y = t.clone()
            for k in range(1, 80):
                w = self.d[:, None] * t
                for s in range(v.shape[0]):
                    w += v[s][:, None] * t[self.idx[s]]
                t = w * (-1j * dt / k)
                y += t
                if float(t.abs().max()) < 1e-18:
                    break
            out[:, c:c + step] = y
        return out

    def step(self, a, dt, P):
        y = self.propagate(a, dt, P)
        return self.propagate(a, dt, y.T.conj().resolve_conj().contiguous()).T.conj().resolve_conj().contiguous()

    def observables(self, a, P):
        return P.diagonal().real.clone(), 2.0 * (self.bond_values(a) * P[self.j, self.i]).imag


def _exact_model(case, rng):
    l1, l2 = case["l1"], case["l2"]
    V = _onsite(case, _sites(case), rng)
    top, T = case["strength"] * _strength_factor(rng), _duration(case)
    ex = _Exact(_lattice_kind(case), l1, l2, _periodic(case), case["field"], _flux_point(case), V, 1.0,
                _lattice_kind(case) == "honeycomb")
    return ex, lambda t: top * (0.3 + 0.7 * t / T)


def _host(x):
    return x.detach().cpu().numpy()


def exact(case, seed):
    rng = np.random.default_rng(seed)
    kind, dt = case["kind"], case.get("dt")
    if kind == "evolve":
        ex, a = _exact_model(case, rng)
        form, x = _initial(ex.n, rng)
        if form == "factor":
            q = torch.from_numpy(x).to(_device())
            P = q @ q.conj().T
        else:
            P = torch.zeros((ex.n, ex.n), dtype=torch.complex128, device=_device())
            P[x, x] = 1.0
        rhos, currents = [], []
        for k in range(case["steps"]):
            P = ex.step(a(k * dt), dt, P)
            if (k + 1) % case["observe"] == 0:
                rho, J = ex.observables(a(k * dt), P)
                rhos.append(_host(rho))
                currents.append(_host(J))
        return {"P": P, "rho": np.array(rhos), "J": np.array(currents)}
    if kind == "batch":
        out = []
        for L in _batch_sides(case):
            V = _onsite(case, L * L, rng)
            occ = np.sort(rng.permutation(L * L)[: L * L // 2])
            ex = _Exact("square", L, L, (False, False), "landau", None, V, 1.0, False)
            P = torch.zeros((L * L, L * L), dtype=torch.complex128, device=_device())
            P[occ, occ] = 1.0
            for _ in range(case["steps"]):
                P = ex.step(case["strength"], dt, P)
            out.append(P)
        return {"P": out, "mean_density": np.array([float(P.diagonal().real.mean()) for P in out])}
    if kind == "krylov":
        lat_xy = _honeycomb_xy(case["l1"], case["l2"])
        V = _krylov_onsite(lat_xy)
        top, T = case["strength"] * _strength_factor(rng), _duration(case)
        ex = _Exact("honeycomb", case["l1"], case["l2"], (False, False), "symmetric", None, V, -2.8, False)
        psi = torch.from_numpy(_random_kets(ex.n, case["kets"], rng)).to(_device())
        rhos = []
        for k in range(case["steps"]):
            psi = ex.propagate(top * (0.3 + 0.7 * k * dt / T), dt, psi)
            rhos.append(_host(psi[:, 0].abs() ** 2))
        psi = _host(psi)
        return {"psi": psi[:, 0].copy() if case["kets"] == 1 else psi, "rho": np.array(rhos)}
    if kind == "kets":
        ex, a = _exact_model(case, rng)
        psi = torch.from_numpy(_random_kets(ex.n, case["kets"], rng)).to(_device())
        for k in range(case["steps"]):
            psi = ex.propagate(a(k * dt), dt, psi)
        last = a((case["steps"] - 1) * dt)
        p = psi[:, 0]
        J = 2.0 * (ex.bond_values(last) * p[ex.j] * p[ex.i].conj()).imag
        return {"psi": _host(psi), "rho": _host(p.abs() ** 2), "J": _host(J)}
    if kind == "gradient":
        return _exact_gradient(case, rng)
    V = _onsite(case, _sites(case), rng)
    ex = _Exact("square", case["l1"], case["l2"], (False, False), "landau", None, V, 1.0, False)
    E, U = np.linalg.eigh(_host(ex.dense(case["strength"] * _strength_factor(rng))))
    f = 1.0 / (np.exp((E - case["mu"]) / case["temperature"]) + 1.0)
    U = torch.from_numpy(U).to(_device())
    return {"P": (U * torch.from_numpy(f).to(_device())) @ U.conj().T}


def _honeycomb_xy(l1, l2):
    j1, j2, b = (x.ravel() for x in np.meshgrid(np.arange(1, l1 + 1), np.arange(1, l2 + 1), np.arange(2), indexing="ij"))
    return np.stack([j1 + 0.5 * j2 + 0.5 * b, math.sqrt(3.0) / 2.0 * j2 + math.sqrt(3.0) / 6.0 * b], axis=-1)


def _exact_gradient(case, rng):
    ex, a = _exact_model(case, rng)
    q = torch.from_numpy(_initial(ex.n, rng)[1]).to(_device())
    sites = _loss_sites(case)
    weights = torch.from_numpy(rng.uniform(0.5, 1.5, len(sites))).to(_device())
    dt, M = case["dt"], case["steps"]
    amps = [torch.tensor(a(k * dt), dtype=torch.float64, device=_device(), requires_grad=True) for k in range(M)]
    d = ex.d.clone().requires_grad_(True)
    Q = q                                  # P = Q Q^H: the factor evolves
    unitaries = []
    for k in range(M):
        H = ex.dense(amps[k], d)
        t = torch.eye(ex.n, dtype=torch.complex128, device=_device())
        U = t
        with torch.no_grad():
            for m in range(1, 24):
                t = (-1j * dt / m) * (H @ t)
                U = U + t
        unitaries.append(U)
        # the propagator applied to the factor, term by term, for the gradient
        t = Q
        for m in range(1, 24):
            t = (-1j * dt / m) * (H @ t)
            Q = Q + t
    rho = (Q.abs() ** 2).sum(dim=1)
    loss = (weights * rho[: len(sites)]).sum()
    loss.backward()
    lam = torch.zeros((ex.n, ex.n), dtype=torch.complex128, device=_device())
    lam[range(len(sites)), range(len(sites))] = weights.to(torch.complex128)
    for U in reversed(unitaries):
        lam = U.conj().T @ lam @ U
    return {"rho": _host(rho), "field": np.array([[float(x.grad)] for x in amps]), "onsite": _host(d.grad), "P0": lam}
