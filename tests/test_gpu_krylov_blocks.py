"""A ket of a block gets the same bits as alone: the recurrences of a block's
kets do not mix, whichever form of the product by H the block's size picks
(nine neighbours: another one above eight kets)."""
import numpy as np
import pytest

import lmhip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["honeycomb", "haldane", "third neighbours"])
@pytest.mark.parametrize("m", [8, 9, 65])
def test_kets_of_a_block_as_alone(kind, m):
    lat = lmhip.SquareLattice(13, 11) if kind == "third neighbours" else lmhip.HoneycombLattice(9, 11)
    n = len(lat)
    rng = np.random.default_rng(n + m)
    V = rng.uniform(-0.5, 0.5, n)
    field = lmhip.SymmetricGauge(0.05)
    H = (lmhip.haldane(lat, 1.0, 0.1, 0.2, V, field=field) if kind == "haldane" else
         lmhip.tightbinding_hamiltonian(lat, V, t2=0.3, t3=0.1, field=field) if kind == "third neighbours" else
         lmhip.tightbinding_hamiltonian(lat, V, field=field))
    ctx = lmhip.Context(0)
    ctx.set_hamiltonian(H)
    solver = lmhip.HIPKrylovExp(ctx=ctx)
    solver.update_solver(H, 0.2)
    psi = rng.normal(size=(n, m)) + 1j * rng.normal(size=(n, m))
    block = lmhip.Kets.from_array(ctx, psi)
    solver.step(block)
    got = block.to_numpy()
    for c in (0, m // 2, m - 1):
        one = lmhip.Kets.from_array(ctx, psi[:, c].copy())
        solver.step(one)
        assert np.array_equal(one.to_numpy().ravel(), got[:, c])
