"""The column kernel (H's rows in registers, or loaded a site ahead) at the
edges of its variants' sizes, against the same Taylor polynomial evaluated by
scipy.sparse from the device-built H: kets (plain stores, a column count that
is no multiple of the groups) at every size, a whole step of a non-Hermitian
matrix (conjugate-transposed stores) at the smaller ones, with one repetition
and with several (s > 1)."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

import lmhip
from lmhip import _lib

pytestmark = pytest.mark.gpu

# sites: 128, 129, 256, 257, 512, 513, 1024, 1025, 2048, 2049, 2304, 2305, 3072, 3073, 3840, 3841, 4096
SQUARE = [(8, 16), (3, 43), (16, 16), (1, 257), (16, 32), (27, 19), (32, 32), (25, 41), (32, 64), (3, 683), (48, 48),
          (5, 461), (48, 64), (7, 439), (60, 64), (23, 167), (64, 64)]
# sites: 256, 258, 2048, 2050, 2560, 2562, 3584, 3586, 5120, 5122
HONEY = [(8, 16), (3, 43), (32, 32), (25, 41), (32, 40), (21, 61), (32, 56), (11, 163), (40, 64), (13, 197)]


def _hamiltonian(kind, l1, l2):
    rng = np.random.default_rng(l1 * 1000 + l2)
    if kind == "square":
        lat = lmhip.SquareLattice(l1, l2)
        V = rng.uniform(-0.5, 0.5, len(lat))
        return lmhip.tightbinding_hamiltonian(lat, V, field=lmhip.SymmetricGauge(0.07))
    if kind == "qwz":
        lat = lmhip.SquareLattice(l1, l2)
        return lmhip.qwz(lat, 1.0, rng.uniform(-0.5, 0.5, len(lat)), field=lmhip.SymmetricGauge(0.07))
    lat = lmhip.HoneycombLattice(l1, l2)
    return lmhip.haldane(lat, 1.0, 0.1, 0.2, rng.uniform(-0.5, 0.5, len(lat)), field=lmhip.SymmetricGauge(0.07))


def _sparse(ctx, H):
    diag, hij = ctx.hamiltonian_entries(H)
    b = H.geometry()[0]
    up = {}
    for i, j, v in zip(b.i, b.j, hij):       # H[i, j] whole, once per pair
        up[(int(i), int(j))] = v
    i = np.array([k[0] for k in up], dtype=int)
    j = np.array([k[1] for k in up], dtype=int)
    v = np.array(list(up.values()), dtype=complex)
    n = H.n
    return sp.csr_matrix((np.concatenate([v, v.conj(), diag]),
                          (np.concatenate([i, j, np.arange(n)]), np.concatenate([j, i, np.arange(n)]))), shape=(n, n))


def _poly(S, X, dt, K, s):
    for _ in range(int(s)):
        y = X
        for k in range(K, 0, -1):
            y = X + (-1j * dt / (s * k)) * (S @ y)
        X = y
    return X


CASES = ([("square", a, b) for a, b in SQUARE] + [("honeycomb", a, b) for a, b in HONEY]
         + [("qwz", 5, 7), ("qwz", 23, 31)])


@pytest.mark.parametrize("dt", [0.05, 2.6])
@pytest.mark.parametrize("kind,l1,l2", CASES)
def test_column_variants_at_their_edges(kind, l1, l2, dt):
    H = _hamiltonian(kind, l1, l2)
    n = H.n
    print("case", kind, l1, l2, dt, flush=True)
    ctx = lmhip.Context(0)
    ctx.set_hamiltonian(H)
    solver = lmhip.HIPExp(ctx=ctx, step_mode=_lib.STEP_FUSED_T)
    rng = np.random.default_rng(n)
    psi = rng.normal(size=(n, 7)) + 1j * rng.normal(size=(n, 7))
    kets = lmhip.Kets.from_array(ctx, psi)
    solver.update_solver(H, dt)
    solver.step(kets)
    K, s = solver.K, solver.s
    assert (s > 1) == (dt > 1)
    S = _sparse(ctx, H)
    # roundings of one term: (z + 3) eps max|y|, times K terms and s repetitions,
    # each term's magnitude at most e^{|H| dt / s} of the input's
    scale = float(np.max(np.abs(psi))) * np.exp(min(8.0, float(abs(S).sum(axis=1).max()) * dt / s))
    tol = 16 * np.finfo(float).eps * K * s * scale
    assert np.max(np.abs(kets.to_numpy() - _poly(S, psi, dt, K, s))) <= tol
    v = ctypes.c_int64()
    _lib.check(lmhip.lib().lmh_get_option(ctx.h, _lib.OPT_FUSED_LAUNCHED, ctypes.byref(v)))
    if dt < 1:
        assert v.value > _lib.FUSED_STRIP
    if n <= 1100:
        P = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
        st = lmhip.DensityMatrix.from_array(ctx, P)
        solver.step(st)
        Y = _poly(S, P, dt, K, s)
        want = _poly(S, Y.conj().T, dt, K, s).conj().T
        tol = 16 * np.finfo(float).eps * 2 * K * s * float(np.max(np.abs(P))) * (scale / float(np.max(np.abs(psi)))) ** 2
        assert np.max(np.abs(st.to_numpy() - want)) <= tol
