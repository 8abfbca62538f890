"""P = V diag(f) V^H at the edges of the product's tiles: sizes around 64 and
128 rows, column counts that are and are not multiples of 4, weights of either
sign.  f(E) = E^2 - 0.3 gives H^2 - 0.3 exactly; a window of the spectrum gives
a projector of that rank that commutes with H.  Tolerances: 64 n eps |H|^2
(the eigensystem's backward error and the sums), likewise for the window."""
import numpy as np
import pytest

import lmhip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1, 1), (1, 2), (1, 5), (7, 9), (8, 8), (5, 13), (1, 127), (8, 16), (3, 43), (10, 20)])
def test_tiles(dims):
    n = dims[0] * dims[1]
    rng = np.random.default_rng(n)
    H = lmhip.tightbinding_hamiltonian(lmhip.SquareLattice(*dims), rng.uniform(-1, 1, n), field=lmhip.SymmetricGauge(0.07))
    ctx = lmhip.Context(0)
    ctx.set_hamiltonian(H)
    diag, hij = ctx.hamiltonian_entries(H)
    b = H.geometry()[0]
    D = np.diag(diag).astype(complex)
    D[b.i, b.j] = hij
    D[b.j, b.i] = hij.conj()
    eig = lmhip.diagonalize(H, ctx=ctx)
    tol = 64 * n * 2.2e-16 * max(np.linalg.norm(D, 2), 1.0) ** 2
    print("case projector tiles n=%d" % n, flush=True)
    P = eig.projector(lambda e: e * e - 0.3).to_numpy()
    assert np.max(np.abs(P - (D @ D - 0.3 * np.eye(n)))) <= tol
    assert np.array_equal(np.triu(P, 1), np.tril(P, -1).conj().T)
    for lo, hi in ((0, 1), (n // 3, n // 3 + 3), (n // 2, n), (0, min(n, 6))):
        hi = min(hi, n)
        w = np.zeros(n)
        w[lo:hi] = 1.0
        P = eig.projector(w).to_numpy()
        assert abs(np.trace(P) - (hi - lo)) <= tol
        assert np.max(np.abs(P @ P - P)) <= tol
        assert np.max(np.abs(P @ D - D @ P)) <= 2 * tol
