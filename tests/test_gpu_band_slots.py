"""Per-term steps of an H with a narrow band and more neighbours than the
banded kernels take (13 .. 16 slots per row): they run on the gather pass, by
default as when it is asked for.  A step of a non-Hermitian matrix and kets
against the same Taylor polynomial by scipy.sparse, the autotuner, the refusal
of the banded passes, and a recorded sweep against the one with the gather
pass set explicitly.  Tolerance as in the strip blocks' test: 64 eps K s
exp(dt |H| / s)^s max|P| a side."""
import numpy as np
import pytest
import scipy.sparse as sp

import lmhip
from lmhip import _lib
from lmhip.lattice import Translation

pytestmark = pytest.mark.gpu


def _banded(n, slots, seed):
    """`slots` neighbours of every inner site, within slots / 2 + 1 sites."""
    rng = np.random.default_rng(seed)
    m = sp.coo_matrix((n, n), dtype=complex)
    for k in range(1, slots // 2 + 1):
        m = m + sp.diags(rng.uniform(0.1, 0.3, n - k) * np.exp(1j * rng.uniform(0, 6, n - k)), k, shape=(n, n))
    if slots % 2:                       # one more each: pairs of runs of k sites
        k = slots // 2 + 1
        i = np.arange(n - k)
        i = i[(i // k) % 2 == 0]
        m = m + sp.coo_matrix((rng.uniform(0.1, 0.3, len(i)) + 0j, (i, i + k)), shape=(n, n))
    m = m.tocsr()
    return (m + m.conj().T + sp.diags(rng.uniform(-1, 1, n))).tocsr()


def _poly(S, X, dt, K, s):
    for _ in range(int(s)):
        y = X
        for k in range(K, 0, -1):
            y = X + (-1j * dt / (s * k)) * (S @ y)
        X = y
    return X


@pytest.mark.parametrize("n", [97, 1300])
@pytest.mark.parametrize("slots", [12, 13, 16, 24])
def test_narrow_band_with_many_neighbours(n, slots):
    S = _banded(n, slots, n + slots)
    H = lmhip.SparseHamiltonian.from_scipy(S)
    ctx = lmhip.Context(0)
    solver = lmhip.HIPExp(ctx=ctx, step_mode=_lib.STEP_PER_PASS)
    ctx.set_hamiltonian(H)
    dt = 0.1
    solver.update_solver(H, dt)
    K, s = solver.K, solver.s
    tol = 64 * 2.2e-16 * K * s * np.exp(dt * abs(S).sum(axis=0).max())
    rng = np.random.default_rng(n)
    psi = rng.normal(size=(n, 3)) + 1j * rng.normal(size=(n, 3))
    kets = lmhip.Kets.from_array(ctx, psi)
    solver.step(kets)
    assert np.max(np.abs(kets.to_numpy().reshape(n, 3) - _poly(S, psi, dt, K, s))) <= tol * np.max(np.abs(psi))
    P = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
    st = lmhip.DensityMatrix.from_array(ctx, P)
    want = P
    for _ in range(2):
        solver.step(st)
        want = _poly(S, _poly(S, want, dt, K, s).conj().T, dt, K, s).conj().T
    assert np.max(np.abs(st.to_numpy() - want)) <= 4 * tol * tol / (64 * 2.2e-16 * K * s) * np.max(np.abs(P))


def test_banded_passes_are_refused_and_the_autotuner_runs():
    S = _banded(300, 16, 5)
    H = lmhip.SparseHamiltonian.from_scipy(S)
    ctx = lmhip.Context(0)
    solver = lmhip.HIPExp(ctx=ctx)
    ctx.set_hamiltonian(H)
    for variant in (2, 3):
        assert _lib.lib().lmh_set_option(ctx.h, _lib.OPT_LEFT_PASS, variant) == _lib.LMH_ERANGE
    solver.update_solver(H, 0.1)
    P = np.random.default_rng(1).normal(size=(300, 300)) + 0j
    st = lmhip.DensityMatrix.from_array(ctx, P)
    assert solver.autotune(st, reps=1)["best_ms"] > 0


def test_recorded_sweep_with_sixteen_slots():
    lat = lmhip.SquareLattice(30, 7)
    n = len(lat)
    hops = [(1, 0), (0, 1), (1, 1), (1, -1), (2, 0), (0, 2), (1, 2), (2, 1)]
    V = np.random.default_rng(3).uniform(-0.5, 0.5, n)

    def h(t):
        return lmhip.construct_hamiltonian(lat, V, *[(0.2, Translation((0, 0), d)) for d in hops],
                                           field=lmhip.SymmetricGauge(0.02 + 0.05 * t))

    out = []
    for left in (None, 1):
        ctx = lmhip.Context(0)
        _lib.check(_lib.lib().lmh_set_option(ctx.h, _lib.OPT_ADJOINT_MODE, 2))
        ctx.set_hamiltonian(h(0.0))
        if left:
            _lib.check(_lib.lib().lmh_set_option(ctx.h, _lib.OPT_LEFT_PASS, left))
        P0 = np.diag((np.arange(n) % 2).astype(complex))
        ev = lmhip.Evolution(lmhip.HIPExp(ctx=ctx, step_mode=_lib.STEP_PER_PASS), h, P0)
        tape = lmhip.EvolutionTape(ev, 2)
        for _ in ev([0.1 * k for k in range(5)]):
            pass
        g = tape.backward(lmhip.localdensity_cotangent(n, 1.0, sites=np.arange(n // 3)))
        out.append((ev.states[0].to_numpy(), g.onsite, g.field, g.P0.to_numpy()))
        tape.close()
    for a, b in zip(*out):
        # four steps of K <= 10 terms and both sides, entries of order n
        assert np.max(np.abs(a - b)) <= 1e-12 * max(1.0, np.max(np.abs(b)))
