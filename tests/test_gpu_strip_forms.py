"""Every form of the strip kernel (block shape, a term in two phases or in one)
on the grids of strip_grids.py: kets and steps of a non-Hermitian matrix
against the same Taylor polynomial by scipy.sparse, real and complex bonds
along x, open and periodic edges, one repetition and several.  Tolerance as in
the strip blocks' test: 64 eps K s exp(dt |H| / s)^s max|P| a side."""
import ctypes

import numpy as np
import pytest

import lmhip
import strip_grids
from lmhip import _lib
from test_gpu_strip_blocks import _csr, _poly

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lx,ly,shape,phases", strip_grids.FORMS)
@pytest.mark.parametrize("periodic", [(False, False), (True, True)])
def test_form(lx, ly, shape, phases, periodic):
    n = lx * ly
    rng = np.random.default_rng(n)
    for xphase, dt in ((False, 0.05), (True, 0.13), (False, 1.1)):
        S = _csr(lx, ly, periodic[0], periodic[1], 3 * n, xphase)
        H = lmhip.SparseHamiltonian.from_scipy(S)
        ctx = lmhip.Context(0)
        solver = lmhip.HIPExp(ctx=ctx, step_mode=_lib.STEP_FUSED_T)
        ctx.set_hamiltonian(H)
        solver.update_solver(H, dt)
        K, s = solver.K, solver.s
        tol = 64 * 2.2e-16 * K * s * np.exp(dt * abs(S).sum(axis=0).max())
        psi = rng.normal(size=(n, 5)) + 1j * rng.normal(size=(n, 5))
        k = lmhip.Kets.from_array(ctx, psi)
        _lib.check(_lib.lib().lmh_kets_step(ctx.h, k.h))
        launched = ctypes.c_int64()
        _lib.check(_lib.lib().lmh_get_option(ctx.h, _lib.OPT_FUSED_LAUNCHED, ctypes.byref(launched)))
        assert launched.value == _lib.FUSED_STRIP
        err = np.max(np.abs(k.to_numpy().reshape(n, 5) - _poly(S, psi, dt, K, s)))
        print("grid %dx%d %s %s dt %g K %d s %g kets %.1e (tol %.1e)" % (lx, ly, periodic, xphase, dt, K, s, err,
                                                                      tol * np.max(np.abs(psi))), flush=True)
        assert err <= tol * np.max(np.abs(psi))
        if n > 1400 and (n > 2700 or not xphase or any(periodic) or shape != (1, 20)):
            continue                             # (the largest are checked by their kets)
        P = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
        st = lmhip.DensityMatrix.from_array(ctx, P)
        want = P
        for _ in range(2):
            solver.step(st)
            want = _poly(S, _poly(S, want, dt, K, s).conj().T, dt, K, s).conj().T
        assert np.max(np.abs(st.to_numpy() - want)) <= 4 * tol * tol / (64 * 2.2e-16 * K * s) * np.max(np.abs(P))
