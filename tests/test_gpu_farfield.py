"""The far field's products at their edges: directions below, at and above the 16 of a
block, spheres at and beyond the 4 of a step and the 128 of a chunk, orders that leave the
last tile of 16 entries partly empty, one sphere far larger than the rest, coefficients
beyond a sphere's order set to NaN (never read), and orders above the 112 up to which the
azimuthal factors are kept.

Reference: the oracle (1e-12 of the largest value, as for a single sphere: recurrences and
phases of a few tens of eps, summed); above order 112 the same coefficients in a context of
lower order."""
import math

import numpy as np
import pytest

from helpers import snm_flat
from itofoggysim_amd import MultiSphereSolver
from oracle import farfield as FF

pytestmark = pytest.mark.gpu


def _setup(ns, lmax, n_global, seed):
    rng = np.random.default_rng(seed)
    g = np.arange(ns)
    pos = (np.stack([g // 36, g // 6 % 6, g % 6], 1) - 3 + rng.uniform(-0.1, 0.1, (ns, 3))) * 2.5
    s = MultiSphereSolver(pos, np.full(ns, 1.0), 1.4, 1.0, lmax=lmax, n_global=n_global)
    S, mask = snm_flat(n_global, lmax)
    x = (rng.standard_normal(s.n) + 1j * rng.standard_normal(s.n)) * mask / S
    return s, pos, x, mask, rng


@pytest.mark.parametrize("ns,ndir,big", [(1, 1, 1), (3, 15, 2), (4, 16, 9), (5, 17, 13), (128, 33, 3), (131, 5, 6)])
def test_against_oracle(ns, ndir, big):
    lmax = np.full(ns, min(2, big), np.int32)
    lmax[ns // 2] = big
    s, pos, x, mask, rng = _setup(ns, lmax, big, ns + ndir)
    th = rng.uniform(0.0, math.pi, ndir)
    ph = rng.uniform(-math.pi, 2 * math.pi, ndir)
    th[0] = 0.0
    ref = np.concatenate(FF.far_field(x, pos, big, 1.0, th, ph))
    got = np.concatenate(s.far_field(np.where(mask, x, np.nan), th, ph))
    s.close()
    err = np.max(np.abs(got - ref)) / np.max(np.abs(ref))
    print(f"{ns} spheres, {ndir} directions, order {big}: {err:.1e}")
    assert err < 1e-12


def test_orders_beyond_the_kept_azimuthal_factors():
    th, ph = np.linspace(0.0, math.pi, 21), np.linspace(-1.0, 6.0, 21)
    out = []
    for N in (100, 131):
        s, pos, x, mask, _ = _setup(3, np.array([100, 7, 30], np.int32), 100, 5)
        if N > 100:
            s.close()
            s = MultiSphereSolver(pos, np.full(3, 1.0), 1.4, 1.0, lmax=[100, 7, 30], n_global=N)
            y = np.full((6, N * (N + 2)), np.nan, complex)
            y[:, :100 * 102] = x.reshape(6, -1)
            x = y.ravel()
        out.append(np.concatenate(s.far_field(x, th, ph)))
        s.close()
    err = np.max(np.abs(out[1] - out[0])) / np.max(np.abs(out[0]))
    print(f"order 131 against 100: {err:.1e}")
    assert err < 1e-12


@pytest.mark.parametrize("N", [112, 113])
def test_last_order_with_kept_azimuthal_factors_and_the_next(N):
    """The factors e^{i m phi} stay in local memory up to order 112: the same coefficients in contexts of
    order N and of order 100."""
    th, ph = np.linspace(0.0, math.pi, 19), np.linspace(-1.0, 6.0, 19)
    lmax = np.array([100, 7, 30], np.int32)
    s, pos, x, _, _ = _setup(3, lmax, 100, 5)
    ref = np.concatenate(s.far_field(x, th, ph))
    s.close()
    s = MultiSphereSolver(pos, np.full(3, 1.0), 1.4, 1.0, lmax=lmax, n_global=N)
    y = np.full((6, N * (N + 2)), np.nan, complex)
    y[:, :100 * 102] = x.reshape(6, -1)
    got = np.concatenate(s.far_field(y.ravel(), th, ph))
    s.close()
    err = np.max(np.abs(got - ref)) / np.max(np.abs(ref))
    print(f"order {N} against 100: {err:.1e}")
    assert err < 1e-12
