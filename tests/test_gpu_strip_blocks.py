"""The blocks of the strip kernel at the edges of their shapes and sizes:
grids that the blocks divide and grids that they do not, sides at, below and
above a block's, one to several columns per workgroup, narrow grids that only
whole strips fit, periodic and open edges, a diagonal disorder, a real and a
complex bond along x, odd and even term counts and s > 1.  A step of a non-Hermitian matrix and a
plain pass over kets, against the same Taylor polynomial by scipy.sparse from
the device-built H.  Tolerance: each of the K terms of a side adds a few
rounding errors of the partial sums, whose size the polynomial's bound
exp(dt |H|) |P| limits: 64 eps K s exp(dt |H| / s)^s max|P|."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

import lmhip
from lmhip import _lib

pytestmark = pytest.mark.gpu

# (lx, ly), periodic (x, y)
GRIDS = [((3, 4), (False, False)), ((2, 5), (False, True)), ((4, 4), (True, True)), ((5, 7), (True, True)),
         ((8, 8), (False, False)), ((7, 12), (True, False)), ((9, 10), (False, True)), ((12, 16), (True, True)),
         ((13, 17), (False, False)), ((37, 23), (False, True)), ((23, 37), (True, False)), ((32, 32), (True, True)),
         ((33, 33), (False, False)), ((44, 44), (False, False)), ((48, 48), (True, True)), ((47, 47), (True, True)),
         ((3, 340), (False, False)), ((5, 400), (False, True)), ((340, 5), (True, False)), ((64, 40), (False, False))]


def _csr(lx, ly, px, py, seed, xphase):
    """A Landau-gauge grid (y bonds by x column), real or complex x bonds."""
    rng = np.random.default_rng(seed)
    n = lx * ly
    i = np.arange(n)
    x, y = i // ly, i % ly
    t = np.exp(1j * rng.uniform(0, 6, lx)) * rng.uniform(0.5, 1.5, lx)
    rows, cols, vals = [], [], []
    up = (y + 1 < ly) | (py and ly >= 3)
    rows.append(i[up]); cols.append((x * ly + (y + 1) % ly)[up]); vals.append(t[x][up])
    u = rng.uniform(0.5, 1.5, lx) * (np.exp(1j * rng.uniform(0, 6, lx)) if xphase else 1.0)
    right = (x + 1 < lx) | (px and lx >= 3)
    rows.append(i[right]); cols.append((((x + 1) % lx) * ly + y)[right]); vals.append((u[x] + 0j)[right])
    r, c, v = np.concatenate(rows), np.concatenate(cols), np.concatenate(vals)
    m = sp.coo_matrix((v, (r, c)), shape=(n, n)).tocsr()
    return (m + m.conj().T + sp.diags(rng.uniform(-1, 1, n))).tocsr()


def _poly(S, X, dt, K, s):
    for _ in range(int(s)):
        y = X
        for k in range(K, 0, -1):
            y = X + (-1j * dt / (s * k)) * (S @ y)
        X = y
    return X


@pytest.mark.parametrize("dims,periodic", GRIDS)
def test_blocks(dims, periodic):
    lx, ly = dims
    n = lx * ly
    rng = np.random.default_rng(n)
    for xphase, dt in ((False, 0.05), (True, 0.13), (False, 1.1)):
        S = _csr(lx, ly, periodic[0], periodic[1], 7 * n, xphase)
        H = lmhip.SparseHamiltonian.from_scipy(S)
        ctx = lmhip.Context(0)
        solver = lmhip.HIPExp(ctx=ctx, step_mode=_lib.STEP_FUSED_T)
        ctx.set_hamiltonian(H)
        solver.update_solver(H, dt)
        K, s = solver.K, solver.s
        tol = 64 * 2.2e-16 * K * s * np.exp(dt * abs(S).sum(axis=0).max())
        launched = ctypes.c_int64()
        m = 5
        psi = rng.normal(size=(n, m)) + 1j * rng.normal(size=(n, m))
        k = lmhip.Kets.from_array(ctx, psi)
        _lib.check(_lib.lib().lmh_kets_step(ctx.h, k.h))
        err = np.max(np.abs(k.to_numpy().reshape(n, m) - _poly(S, psi, dt, K, s)))
        print("grid %s %s x %s dt %g K %d s %g kets %.1e (tol %.1e)" % (dims, periodic, "complex" if xphase else "real",
                                                                     dt, K, s, err, tol * np.max(np.abs(psi))), flush=True)
        assert err <= tol * np.max(np.abs(psi))
        if n > 2400:
            continue
        P = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
        st = lmhip.DensityMatrix.from_array(ctx, P)
        want = P
        for _ in range(2):
            solver.step(st)
            left = _poly(S, want, dt, K, s)
            want = _poly(S, left.conj().T, dt, K, s).conj().T
        _lib.check(_lib.lib().lmh_get_option(ctx.h, _lib.OPT_FUSED_LAUNCHED, ctypes.byref(launched)))
        err = np.max(np.abs(st.to_numpy() - want))
        print("   step: variant %d err %.1e" % (launched.value, err), flush=True)
        assert launched.value == _lib.FUSED_STRIP
        assert err <= 4 * tol * tol / (64 * 2.2e-16 * K * s) * np.max(np.abs(P))
