"""The per-term schedule chosen where the caller sets none, against the column
sweep (right pass 3, single-term left passes) set explicitly: the same U P U'
to rounding, for a P that is not Hermitian, read after odd and even numbers of
steps (the default leaves the state in its conjugate-transposed form)."""
import numpy as np
import pytest

import lmhip
from lmhip import _lib

pytestmark = pytest.mark.gpu


def _lattice(kind):
    if kind == "square":
        return lmhip.SquareLattice(9, 13)
    if kind == "honeycomb":
        return lmhip.HoneycombLattice(7, 11)
    # periodic: the band is wider than the banded passes take
    return lmhip.HoneycombLattice(24, 24, boundaries=(("axis1", True),))


@pytest.mark.parametrize("kind", ["square", "honeycomb", "wide band"])
@pytest.mark.parametrize("steps", [1, 2, 3])
def test_default_schedule_is_the_column_sweep_to_rounding(kind, steps):
    lat = _lattice(kind)
    n = len(lat)
    rng = np.random.default_rng(n + steps)
    V = rng.uniform(-0.5, 0.5, n)
    P = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))

    def h(t):
        f = lmhip.SymmetricGauge(0.01 + 0.02 * t)
        return (lmhip.haldane(lat, 1.0, 0.1, 0.2, V, field=f) if kind != "square"
                else lmhip.tightbinding_hamiltonian(lat, V, field=f))

    out = []
    for explicit in (True, False):
        ctx = lmhip.Context(0)
        solver = lmhip.HIPExp(ctx=ctx, step_mode=_lib.STEP_PER_PASS)
        if explicit:
            _lib.check(lmhip.lib().lmh_set_option(ctx.h, _lib.OPT_RIGHT_PASS, 3))
            _lib.check(lmhip.lib().lmh_set_option(ctx.h, _lib.OPT_LEFT_PASS, 1))
        ev = lmhip.Evolution(solver, h, P)
        for _ in ev([0.05 * k for k in range(steps + 1)]):
            pass
        rho, J = lmhip.observables(ev.states[0])
        out.append((rho, J, ev.states[0].to_numpy()))
    # K <= 10 terms and both sides of each step: a few hundred roundings of
    # entries up to max |P|
    tol = 1e-13 * steps * float(np.max(np.abs(P)))
    for a, b in zip(*out):
        assert np.max(np.abs(a - b)) <= tol
