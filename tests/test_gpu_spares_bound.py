"""Buffers that destroyed states leave with their context: kept for the next
state whatever smaller ones were left before, and given back on request."""
import numpy as np
import pytest
import torch

import lmhip

pytestmark = pytest.mark.gpu

SIDE = 40                                   # N = 1600: 41 MB a buffer, three a state
STATE = 3 * 16 * SIDE ** 4


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info(0)[0]


def _hamiltonian():
    return lmhip.tightbinding_hamiltonian(lmhip.SquareLattice(SIDE, SIDE), field=lmhip.LandauGauge(0.01))


def test_small_buffers_make_room_for_large_ones():
    H, n = _hamiltonian(), SIDE * SIDE
    ctx = lmhip.Context(0)
    ctx.set_hamiltonian(H)
    krylov = lmhip.HIPKrylovExp(ctx=ctx)
    krylov.update_solver(H, 0.1)
    rng = np.random.default_rng(0)
    for m in (1, 2, 3, 4, 5):               # seven buffers each
        k = lmhip.Kets.from_array(ctx, rng.normal(size=(n, m)) + 0j)
        krylov.step(k)
        k.close()
    before = _free()
    lmhip.DensityMatrix(ctx, n).close()
    kept = before - _free()
    assert 0.9 * STATE <= kept              # its three buffers wait for the next state
    P = lmhip.DensityMatrix(ctx, n)
    assert abs(before - _free() - kept) <= 0.1 * STATE
    P.close()
    ctx.close()


def test_spares_are_given_back_on_request():
    H, n = _hamiltonian(), SIDE * SIDE
    a, b = lmhip.Context(0), lmhip.Context(0)
    for ctx in (a, b):
        ctx.set_hamiltonian(H)
    before = _free()
    for ctx in (a, b):
        lmhip.DensityMatrix(ctx, n).close()
    assert before - _free() >= 1.9 * STATE
    a.release_spares()
    assert 0.9 * STATE <= before - _free() <= 1.1 * STATE
    lmhip._lib.check(lmhip.lib().lmh_release_spares(None))
    assert before - _free() <= 0.1 * STATE
    # and the contexts go on
    P = lmhip.DensityMatrix.from_array(a, np.eye(n, dtype=complex))
    assert np.array_equal(P.to_numpy(), np.eye(n))
