"""Gram-Schmidt of the Krylov solvers: sums over one block's slice and over several, vector
counts below, at and above the four that share a read of the new vector.

Reference: the smallest ||b - M x|| over the same Krylov space, from a least-squares problem
in NumPy with products by the solver under test.  A backward stable GMRES of m steps reaches
it to about m sqrt(n) eps ||b|| <= 30 * 120 * 1.1e-16 = 4e-13: 1e-12 here."""
import numpy as np
import pytest

from helpers import snm_flat
from itofoggysim_amd import MultiSphereSolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns,lmax,steps", [(2, 1, 1), (3, 5, 4), (5, 9, 5), (40, 12, 9), (40, 12, 30)])
def test_steps_reach_the_least_squares_minimum(ns, lmax, steps):
    rng = np.random.default_rng(ns + steps)
    g = np.arange(ns)
    pos = (np.stack([g // 16, g // 4 % 4, g % 4], 1) + rng.uniform(-0.1, 0.1, (ns, 3))) * 3.0 * lmax
    lm = np.full(ns, lmax, np.int32)
    s = MultiSphereSolver(pos, 0.8 * lm, 1.5 + 0.1j, 1.0, lmax=lm)
    S, _ = snm_flat(s.n_global, lm)
    R = (rng.standard_normal((3, s.n)) + 1j * rng.standard_normal((3, s.n))) / S
    kw = dict(restart=steps, max_iter=steps, tol=1e-300, raise_on_noconv=False)
    single = [s.solve(b, **kw) for b in R]
    X, infos = s.solve_batch(R, **kw)
    for r in range(3):
        b = R[r] * S
        nb = np.linalg.norm(b)
        V, W = [b / nb], []
        for _ in range(steps):
            W.append(s.calculate_vector_b(V[-1] / S) * S)
            w = W[-1].copy()
            for _ in range(2):
                for v in V:
                    w -= np.vdot(v, w) * v
            V.append(w / np.linalg.norm(w))
        K = np.stack(W, 1)
        best = np.linalg.norm(b - K @ np.linalg.lstsq(K, b, rcond=None)[0]) / nb
        for x, info in (single[r], (X[r], infos[r])):
            got = np.linalg.norm(b - s.calculate_vector_b(x) * S) / nb
            print(f"{ns} spheres, {steps} steps, rhs {r}: residual {got:.12e}, smallest {best:.12e}")
            assert abs(got - best) < 1e-12 and abs(info["rel_residual"] - got) < 1e-12
    s.close()
