"""The order of the Lanczos kernels' sums: a block of 256 rows by halves (128,
64, ..., 1), then the blocks' partials, thread t those of t, t + 256, ..., by
halves again.  With H = 0 a step of a real ket is (psi / |psi|) |psi|, each
factor rounded once, so its bits show which |psi| the kernels found."""
import numpy as np
import pytest

import lmhip

pytestmark = pytest.mark.gpu


def _halves(v):
    v = v.copy()
    while len(v) > 1:
        v = v[: len(v) // 2] + v[len(v) // 2:]
    return v[0]


def _norm(x):
    sq = np.zeros((len(x) + 255) // 256 * 256)
    sq[: len(x)] = x * x
    part = [_halves(b) for b in sq.reshape(-1, 256)]
    acc = np.zeros(256)
    for k, p in enumerate(part):
        acc[k % 256] += p
    return np.sqrt(_halves(acc))


@pytest.mark.parametrize("n,m", [(16, 1), (255, 1), (257, 3), (4000, 1), (65536, 2), (70000, 1)])
def test_norm_of_a_ket_is_summed_by_halves(n, m):
    lat = lmhip.SquareLattice(n // 16 if n % 16 == 0 else 1, 16 if n % 16 == 0 else n)
    H = lmhip.construct_hamiltonian(lat, np.zeros(n))
    ctx = lmhip.Context(0)
    solver = lmhip.HIPKrylovExp(ctx=ctx)
    rng = np.random.default_rng(n)
    for _ in range(4):
        psi = rng.normal(size=(n, m))
        ctx.set_hamiltonian(H)
        kets = lmhip.Kets.from_array(ctx, psi.astype(complex))
        solver.update_solver(H, 0.1)
        solver.step(kets)
        got = kets.to_numpy().reshape(n, m)
        for c in range(m):
            beta = _norm(psi[:, c])
            assert np.array_equal(got[:, c].real, (psi[:, c] * (1.0 / beta)) * beta)
            assert not got[:, c].imag.any()
