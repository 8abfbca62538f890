"""Which per-term steps take two Horner terms per launch: those of an H with at
most 9 slots per row (10 .. 12 run single banded terms).  The launches of a
step are counted by the profile; K terms a side."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

import lmhip
from lmhip import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slots,pairs", [(4, True), (8, True), (10, False), (12, False)])
def test_two_terms_per_launch_up_to_nine_slots(slots, pairs):
    n = 200
    rng = np.random.default_rng(slots)
    m = sp.diags([rng.uniform(0.1, 0.3, n - k) + 0j for k in range(1, slots // 2 + 1)], range(1, slots // 2 + 1), shape=(n, n))
    S = (m + m.conj().T + sp.diags(rng.uniform(-1, 1, n))).tocsr()
    H = lmhip.SparseHamiltonian.from_scipy(S)
    ctx = lmhip.Context(0)
    solver = lmhip.HIPExp(ctx=ctx, step_mode=_lib.STEP_PER_PASS)
    ctx.set_hamiltonian(H)
    solver.update_solver(H, 0.1)
    K = solver.K
    st = lmhip.DensityMatrix.from_array(ctx, np.eye(n, dtype=complex))
    _lib.check(_lib.lib().lmh_set_profiling(ctx.h, 1))
    solver.step(st)
    launches, ms = ctypes.c_int64(), ctypes.c_double()
    _lib.check(_lib.lib().lmh_get_profile(ctx.h, _lib.KERNEL_HORNER_LEFT, ctypes.byref(launches), ctypes.byref(ms)))
    assert solver.s == 1 and launches.value == 2 * ((K + 1) // 2 if pairs else K)
    # U P U' of the unit matrix: unitary to the order's threshold
    assert np.max(np.abs(st.to_numpy() - np.eye(n))) <= 1e-9
