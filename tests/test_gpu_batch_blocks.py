"""A batch gives its members' grids the blocks that suit its own launch: the
members, other states of their contexts (with a deferred pass at the time) and
steps of the contexts after the batch go on as if it had not.  Against the same
evolutions in contexts of their own; a step's few hundred roundings of entries
of order one."""
import ctypes

import numpy as np
import pytest

import lmhip
from lmhip import _lib

pytestmark = pytest.mark.gpu

GRIDS = [(35, 35), (2, 300), (23, 37), (3, 340), (24, 24), (400, 5)]


def _h(lx, ly, seed):
    lat = lmhip.SquareLattice(lx, ly)
    V = np.random.default_rng(seed).uniform(-0.5, 0.5, lx * ly)
    return lambda t: lmhip.tightbinding_hamiltonian(lat, V, field=lmhip.LandauGauge(0.03 + 0.1 * t))


def _p0(n, seed):
    q = np.linalg.qr(np.random.default_rng(seed).normal(size=(n, 9)) + 1j)[0]
    return q @ q.conj().T


def _solo(h, P, times):
    ev = lmhip.Evolution(lmhip.HIPExp(ctx=lmhip.Context(0)), h, P)
    for _ in ev(times):
        pass
    return ev.states[0].to_numpy()


@pytest.mark.parametrize("moving", [False, True])
def test_uniform_and_mixed_batches(moving):
    hs = [_h(lx, ly, k) for k, (lx, ly) in enumerate(GRIDS)]
    if not moving:
        hs = [(lambda f: (lambda t: f(0.0)))(h) for h in hs]
    Ps = [_p0(lx * ly, k) for k, (lx, ly) in enumerate(GRIDS)]
    batch = lmhip.BatchedEvolution([(h if moving else h(0.0), P) for h, P in zip(hs, Ps)], 0.05)
    assert batch.member_kernels() == [_lib.FUSED_STRIP] * len(GRIDS)
    for _ in range(2):
        batch.step(2)
    times = [0.05 * k for k in range(5)]
    for h, P, st in zip(hs, Ps, batch.states):
        assert np.max(np.abs(st.to_numpy() - _solo(h, P, times))) <= 1e-13
    batch.close()


@pytest.mark.parametrize("lx,ly", [(35, 35), (25, 100)])
def test_other_states_of_a_members_context(lx, ly):
    n, h = lx * ly, _h(lx, ly, 7)
    H = h(0.0)
    ctx = lmhip.Context(0)
    solver = lmhip.HIPExp(ctx=ctx)
    P, Q = _p0(n, 1), _p0(n, 2)
    ctx.set_hamiltonian(H)
    a, b = lmhip.DensityMatrix.from_array(ctx, P), lmhip.DensityMatrix.from_array(ctx, Q)
    solver.update_solver(H, 0.05)
    solver.step(b)
    solver.step(b)                                  # its second pass is deferred
    handle = ctypes.c_void_p()
    L = _lib.lib()
    _lib.check(L.lmh_batch_create(ctypes.byref(handle), 1, (ctypes.c_void_p * 1)(ctx.h.value),
                                  (ctypes.c_void_p * 1)(a.h.value)))
    _lib.check(L.lmh_batch_step(handle, 3, 1))
    solver.step(b)
    _lib.check(L.lmh_batch_step(handle, 1, 0))
    _lib.check(L.lmh_batch_destroy(handle))
    solver.step(a)
    solver.update_solver(h(0.4), 0.05)
    solver.step(b)
    static, later = (lambda t: H), (lambda t: H if t < 0.15 - 1e-9 else h(0.4))
    assert np.max(np.abs(a.to_numpy() - _solo(static, P, [0.05 * k for k in range(6)]))) <= 1e-13
    assert np.max(np.abs(b.to_numpy() - _solo(later, Q, [0.05 * k for k in range(5)]))) <= 1e-13


def test_a_second_batch_of_a_context_may_change_its_blocks():
    """The first is too small for the batch's blocks; its tables follow."""
    lx, ly = 2, 300
    n, h = lx * ly, _h(lx, ly, 3)
    H = h(0.0)
    L = _lib.lib()
    ctxs, solvers, first, second = [], [], None, []
    for r in range(6):
        ctx = lmhip.Context(0)
        ctx.set_hamiltonian(H)
        solver = lmhip.HIPExp(ctx=ctx)
        solver.update_solver(H, 0.05)
        ctxs.append(ctx)
        solvers.append(solver)
        second.append(lmhip.DensityMatrix.from_array(ctx, _p0(n, 10 + r)))
    first = lmhip.DensityMatrix.from_array(ctxs[0], _p0(n, 1))

    def create(cs, states):
        handle = ctypes.c_void_p()
        _lib.check(L.lmh_batch_create(ctypes.byref(handle), len(cs), (ctypes.c_void_p * len(cs))(*[c.h.value for c in cs]),
                                      (ctypes.c_void_p * len(cs))(*[s.h.value for s in states])))
        return handle

    a = create(ctxs[:1], [first])
    _lib.check(L.lmh_batch_step(a, 2, 0))
    b = create(ctxs, second)
    _lib.check(L.lmh_batch_step(b, 2, 0))
    _lib.check(L.lmh_batch_step(a, 2, 0))
    _lib.check(L.lmh_batch_step(b, 1, 0))
    times = [0.05 * k for k in range(5)]
    assert np.max(np.abs(first.to_numpy() - _solo(lambda t: H, _p0(n, 1), times))) <= 1e-13
    for r, st in enumerate(second):
        assert np.max(np.abs(st.to_numpy() - _solo(lambda t: H, _p0(n, 10 + r), times[:4]))) <= 1e-13
    for handle in (a, b):
        _lib.check(L.lmh_batch_destroy(handle))
