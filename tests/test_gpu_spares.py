"""Buffers of destroyed states are used again by the context's next states:
the evolutions that follow must not see anything of the ones before."""
import numpy as np
import pytest

import lmhip

pytestmark = pytest.mark.gpu


def _run(ctx, n, field, taped, P0):
    lat = lmhip.SquareLattice(n, n)
    h = lambda t: lmhip.tightbinding_hamiltonian(lat, np.linspace(-0.5, 0.5, n * n), field=field(0.05 + 0.1 * t))
    ctx.set_hamiltonian(h(0.0))
    ev = lmhip.Evolution(lmhip.HIPExp(ctx=ctx), h, P0)
    tape = lmhip.EvolutionTape(ev, 2) if taped else None
    for _ in ev([0.05 * k for k in range(5)]):
        pass
    out = [ev.states[0].to_numpy()]
    if taped:
        g = tape.backward(lmhip.localdensity_cotangent(n * n, 1.0, sites=np.arange(n)))
        tape.close()
        out += [g.onsite, g.field, g.P0.to_numpy()]
    return out


@pytest.mark.parametrize("field", [lmhip.LandauGauge, lambda a: lmhip.PointFlux(a, (4.5, 4.5))])
@pytest.mark.parametrize("taped", [False, True])
def test_reused_buffers_hold_nothing_of_their_past(field, taped):
    rng = np.random.default_rng(5)
    states = []
    for n in (9, 9, 12, 9):
        q = np.linalg.qr(rng.normal(size=(n * n, 6)) + 1j * rng.normal(size=(n * n, 6)))[0]
        states.append((n, q @ q.conj().T))
    shared = lmhip.Context(0)
    for n, P0 in states:             # a size change in between
        got = _run(shared, n, field, taped, P0)
        want = _run(lmhip.Context(0), n, field, taped, P0)
        for a, b in zip(got, want):
            assert np.array_equal(a, b)


def test_kets_and_states_share_the_spares():
    lat = lmhip.SquareLattice(8, 8)
    h = lambda t: lmhip.tightbinding_hamiltonian(lat, field=lmhip.PointFlux(0.1 + t, (4.5, 4.5)))
    rng = np.random.default_rng(6)
    psi = rng.normal(size=(64, 64)) + 1j * rng.normal(size=(64, 64))
    def block(ctx):
        ctx.set_hamiltonian(h(0.0))
        ev = lmhip.Evolution(lmhip.HIPKrylovExp(ctx=ctx), h, lmhip.Kets.from_array(ctx, psi))
        for _ in ev([0.0, 0.1, 0.2]):
            pass
        return ev.states[0].to_numpy()
    shared = lmhip.Context(0)
    want = block(shared)
    _run(shared, 8, lmhip.LandauGauge, False, psi @ psi.conj().T)
    assert np.array_equal(block(shared), want)
