"""The Lanczos kernels at the edges of their sizes, against the exact
propagator (scipy.linalg.expm of the oracle's Hamiltonian): one row, row counts
around a workgroup and around twice a workgroup, each width of the product
(up to 4, 9 and 16 neighbours), 64 and 65 kets (the coefficients written to the
host by the kernel, or copied), and steps of up to 64 and of more basis vectors
(the combination's coefficients as arguments, or uploaded).  The bar is the
propagator's own, 1e-10."""
import ctypes

import numpy as np
import pytest
import scipy.linalg as sl
import scipy.sparse as sp

import lmhip
from lmhip import _lib

pytestmark = pytest.mark.gpu

TOL = 1e-10


def _matrix(n, hops, seed):
    rng = np.random.default_rng(seed)
    m = sp.diags(rng.uniform(-0.5, 0.5, n)).astype(complex)
    for o in range(1, hops + 1):
        if o < n:
            v = np.exp(2j * np.pi * rng.uniform(size=n - o)) * rng.uniform(0.3, 1.0, n - o)
            u = sp.diags(v, o, shape=(n, n))
            m = m + u + u.conj().T
    return m.tocsr()


@pytest.mark.parametrize("n,hops,nkets,dt,dim", [
    (1, 1, 1, 0.3, 30), (255, 2, 1, 0.1, 30), (256, 2, 2, 0.1, 30), (257, 1, 1, 0.1, 30), (511, 4, 1, 0.1, 30),
    (513, 3, 3, 0.1, 30), (300, 8, 1, 0.05, 30), (300, 6, 65, 0.05, 30), (200, 2, 64, 0.1, 30), (90, 1, 65, 0.1, 30),
    (400, 2, 1, 9.0, 63), (400, 2, 1, 9.0, 64), (400, 2, 1, 14.0, 100), (400, 2, 2, 14.0, 100)])
def test_edges(n, hops, nkets, dt, dim):
    print("case krylov edge", n, hops, nkets, dt, dim, flush=True)
    S = _matrix(n, hops, n + hops)
    H = lmhip.SparseHamiltonian.from_scipy(S)
    rng = np.random.default_rng(3)
    psi = rng.normal(size=(n, nkets)) + 1j * rng.normal(size=(n, nkets))
    psi /= np.linalg.norm(psi, axis=0)
    ctx = lmhip.Context(0)
    U = sl.expm(-1j * dt * S.toarray())
    for graphs in (1, 0):
        _lib.check(_lib.lib().lmh_set_option(ctx.h, _lib.OPT_KRYLOV_GRAPHS, graphs))
        ctx.set_hamiltonian(H)
        k = lmhip.Kets.from_array(ctx, psi)
        exact = psi
        for _ in range(3):
            mv = ctypes.c_int64()
            _lib.check(_lib.lib().lmh_krylov_step(ctx.h, k.h, dt, dim, 1e-13, 100, ctypes.byref(mv)))
            exact = U @ exact
            worst = float(np.max(np.abs(k.to_numpy().reshape(n, nkets) - exact)))
            print("  graphs %d matvecs %d worst %.2e" % (graphs, mv.value, worst), flush=True)
            assert worst <= TOL
