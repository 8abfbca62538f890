"""Where the fused pass of an H with 5 to 9 neighbours runs the column kernel
and where the general one, by size and neighbours, and the kernel of the
largest sizes up to its last row (10240 sites, one column in all of the LDS).
Kets against the same Taylor polynomial by scipy.sparse; tolerance as in the
column kernel's test: (z + 3) roundings a term, 16 eps K s e^(|H| dt / s)."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

import lmhip
from lmhip import _lib
from lmhip.lattice import Translation

pytestmark = pytest.mark.gpu

GENERAL_3072, GENERAL_5120 = 18, 14
COLUMN0 = _lib.FUSED_STRIP + 1


def _hamiltonian(slots, l1, l2):
    rng = np.random.default_rng(l1 * 1000 + l2)
    lat = lmhip.HoneycombLattice(l1, l2) if slots in (5, 7, 9) else lmhip.SquareLattice(l1, l2)
    V = rng.uniform(-0.5, 0.5, len(lat))
    field = lmhip.SymmetricGauge(0.03)
    if slots == 9:
        return lmhip.haldane(lat, 1.0, 0.1, 0.2, V, field=field)
    if slots == 8:
        return lmhip.tightbinding_hamiltonian(lat, V, t2=0.3, field=field)
    if slots == 6:
        hops = [Translation((0, 0), d) for d in ((1, 0), (0, 1), (1, 1))]
    else:
        hops = lat.nn_shell(1) + [Translation((0, 0), d) for d in ((1, 0), (0, 1))[:(slots - 3) // 2]]
    return lmhip.construct_hamiltonian(lat, V, *[(0.5 + 0.1 * k, t) for k, t in enumerate(hops)], field=field)


def _sparse(ctx, H):
    diag, hij = ctx.hamiltonian_entries(H)
    b = H.geometry()[0]
    up = {}
    for i, j, v in zip(b.i, b.j, hij):
        up[(int(i), int(j))] = v
    i = np.array([k[0] for k in up], dtype=int)
    j = np.array([k[1] for k in up], dtype=int)
    v = np.array(list(up.values()), dtype=complex)
    return sp.csr_matrix((np.concatenate([v, v.conj(), diag]),
                          (np.concatenate([i, j, np.arange(H.n)]), np.concatenate([j, i, np.arange(H.n)]))),
                         shape=(H.n, H.n))


# (slots, sides, the variant of a density matrix or of 600 kets, that of a few kets)
@pytest.mark.parametrize("slots,l1,l2,variant,few", [
    (5, 35, 35, COLUMN0 + 16, COLUMN0 + 16), (5, 36, 36, COLUMN0 + 18, COLUMN0 + 18),
    (5, 43, 43, COLUMN0 + 19, COLUMN0 + 19), (5, 46, 46, GENERAL_5120, COLUMN0 + 19),
    (6, 51, 51, GENERAL_3072, COLUMN0 + 18), (6, 64, 64, COLUMN0 + 19, COLUMN0 + 19),
    (6, 17, 241, GENERAL_5120, COLUMN0 + 19), (7, 43, 43, GENERAL_5120, COLUMN0 + 19),
    (7, 23, 90, GENERAL_5120, GENERAL_5120), (8, 50, 50, COLUMN0 + 16, COLUMN0 + 16),
    (8, 13, 197, GENERAL_3072, COLUMN0 + 18), (8, 48, 64, GENERAL_3072, COLUMN0 + 18),
    (8, 7, 439, COLUMN0 + 18, COLUMN0 + 18), (8, 56, 64, COLUMN0 + 18, COLUMN0 + 18),
    (8, 5, 717, GENERAL_5120, GENERAL_5120), (8, 64, 80, GENERAL_5120, GENERAL_5120),
    (8, 3, 1707, COLUMN0 + 20, COLUMN0 + 20), (9, 32, 41, COLUMN0 + 17, COLUMN0 + 18),
    (9, 13, 101, GENERAL_3072, COLUMN0 + 18), (9, 32, 48, GENERAL_3072, COLUMN0 + 18),
    (9, 40, 40, COLUMN0 + 18, COLUMN0 + 18), (9, 50, 50, COLUMN0 + 19, COLUMN0 + 19),
    (9, 71, 69, COLUMN0 + 20, COLUMN0 + 20), (9, 64, 80, COLUMN0 + 20, COLUMN0 + 20)])
@pytest.mark.parametrize("m", [7, 600])
def test_fused_pass_by_size_and_neighbours(slots, l1, l2, variant, few, m):
    H = _hamiltonian(slots, l1, l2)
    n, dt = H.n, 0.05
    print("case", slots, l1, l2, n, m, flush=True)
    ctx = lmhip.Context(0)
    ctx.set_hamiltonian(H)
    solver = lmhip.HIPExp(ctx=ctx, step_mode=_lib.STEP_FUSED_T)
    rng = np.random.default_rng(n)
    psi = rng.normal(size=(n, m)) + 1j * rng.normal(size=(n, m))
    kets = lmhip.Kets.from_array(ctx, psi)
    solver.update_solver(H, dt)
    solver.step(kets)
    K = solver.K
    S = _sparse(ctx, H)
    assert solver.s == 1 and np.max(np.diff(S.indptr)) == slots + 1
    y = psi
    for k in range(K, 0, -1):
        y = psi + (-1j * dt / k) * (S @ y)
    scale = float(np.max(np.abs(psi))) * np.exp(min(8.0, float(abs(S).sum(axis=1).max()) * dt))
    assert np.max(np.abs(kets.to_numpy() - y)) <= 16 * np.finfo(float).eps * K * scale
    v = ctypes.c_int64()
    _lib.check(lmhip.lib().lmh_get_option(ctx.h, _lib.OPT_FUSED_LAUNCHED, ctypes.byref(v)))
    assert v.value == (few if m == 7 else variant)
