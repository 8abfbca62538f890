"""The Taylor-order search at the edges of its kernels: K and s are those of
the oracle's rule, exactly.  Grids around the reach of the two diamonds (9 and
11 hops), periodic ones narrower than the diamond, and single rows; matrices
of 1 to 13 neighbours per site (the row kernel's three widths, and the table
kernel above 12) whose neighbourhoods hold at most, exactly and more than the
256 sites of the first table; a nztol above the threshold, and nztol = 0."""
import sys

import numpy as np
import pytest
import scipy.sparse as sp

import lmhip
from helpers import Model
from oracle import numerics as ON

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


TOLS = [(1e-10, 1e-14), (1e-5, 1e-14), (1e-10, 0.0), (1e-8, 1e-7)]


@pytest.mark.parametrize("dims,periodic", [((1, 1), (False, False)), ((1, 7), (False, False)), ((2, 2), (False, False)),
                                           ((3, 5), (False, True)), ((12, 25), (True, True)), ((17, 19), (True, True)),
                                           ((21, 23), (True, False)), ((30, 31), (False, False))])
def test_grids(dims, periodic):
    m = Model("square", dims, periodic, onsite=np.random.default_rng(5).uniform(-0.5, 0.5, dims[0] * dims[1]))
    spec = [("landau", 0.013, 0, 0)]
    Hd, Ho = m.device_h(spec), m.oracle_h(spec)
    solver = lmhip.HIPExp()
    for dt in (0.003, 0.06, 0.1, 0.17, 0.25, 0.5, 1.3):     # K from 3 to beyond both diamonds
        for thr, nz in TOLS:
            solver.threshold, solver.nztol = thr, nz
            solver.update_solver(Hd, dt, force=True)
            _U, K, s, _d = ON.myexp(Ho, dt, threshold=thr, nztol=nz)
            say("grid %s %s dt=%g thr=%g nz=%g K=%d s=%g" % (dims, periodic, dt, thr, nz, K, s))
            assert (solver.K, solver.s) == (K, s)


class _Oracle:
    def __init__(self, H):
        self.n, self.csc = H.n, H


def _ring(n, offsets, seed):
    """n sites on a ring, each coupled to the sites at the given offsets."""
    rng = np.random.default_rng(seed)
    i = np.concatenate([np.arange(n)] * len(offsets))
    j = np.concatenate([(np.arange(n) + o) % n for o in offsets])
    v = np.exp(2j * np.pi * rng.uniform(size=len(i))) * rng.uniform(0.3, 1.0, len(i))
    m = sp.coo_matrix((v, (i, j)), shape=(n, n)).tocsr()
    m = m + m.conj().T + sp.diags(rng.uniform(-0.5, 0.5, n))
    return lmhip.SparseHamiltonian.from_scipy(m)


@pytest.mark.parametrize("n,offsets", [(2, [1]), (64, [1]), (97, [1, 9]), (255, [1, 16]), (256, [1, 16]), (257, [1, 16]),
                                       (300, [1, 17, 40]), (255, [1, 7, 30, 64]), (256, [1, 7, 30, 64]),
                                       (257, [1, 7, 30, 64]), (128, [64, 1, 2, 3, 4]), (401, [1, 5, 20, 70]),
                                       (256, [1, 3, 9, 27, 81, 101]), (257, [1, 3, 9, 27, 81, 101]),
                                       (256, [128, 1, 3, 9, 27, 81, 101]), (257, [1, 2, 3, 4, 5, 6, 7])])
def test_rings(n, offsets):
    H = _ring(n, offsets, n + len(offsets))
    solver = lmhip.HIPExp()
    for dt in (0.01, 0.1, 0.4, 1.1):
        for thr, nz in TOLS:
            solver.threshold, solver.nztol = thr, nz
            solver.update_solver(H, dt, force=True)
            _U, K, s, _d = ON.myexp(_Oracle(H), dt, threshold=thr, nztol=nz)
            say("ring %d x%d dt=%g thr=%g nz=%g K=%d s=%g" % (n, len(offsets), dt, thr, nz, K, s))
            assert (solver.K, solver.s) == (K, s)
