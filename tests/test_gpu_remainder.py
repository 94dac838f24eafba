"""The last degrees of near box translations (class products next to the plane waves) over
boxes whose size runs through a range of order and distance, so that translations with one
to some tens of last degrees occur, in numbers that leave their column blocks partly empty,
one and three right-hand sides; FP64 against the class products of all degrees (1e-11 as for
the box translations), mixed against FP64 (FP32 products of at most 2 L = 300 terms:
300 * 6e-8 = 2e-5 of the translated part)."""
import numpy as np
import pytest

from helpers import snm_flat
from itofoggysim_amd import MultiSphereSolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side", [110.0, 135.0, 160.0, 190.0, 225.0])
def test_last_degrees(side):
    rng = np.random.default_rng(int(side))
    n = 260
    pos = rng.uniform(0.0, side, (n, 3))
    lmax = rng.integers(1, 5, n).astype(np.int32)
    args = (pos, 0.9 * lmax, 1.4 + 0.01j, 1.0)
    f = MultiSphereSolver(*args, lmax=lmax, use_fmm=True, leaf_size=8)
    d = MultiSphereSolver(*args, lmax=lmax, use_fmm=True, leaf_size=8, workspace_mb=4)
    S, mask = snm_flat(f.n_global, lmax)
    X = np.stack([(rng.standard_normal(f.n) + 1j * rng.standard_normal(f.n)) * mask for _ in range(3)])
    f.profile(True), d.profile(True)
    got, ref = f.calculate_vector_b(X[0] / S) * S, d.calculate_vector_b(X[0] / S) * S
    ran, ref_ran = f.profile_read(), d.profile_read()
    f.profile(False), d.profile(False)
    batch, ref_batch = f.calculate_vector_b_batch(X / S) * S, d.calculate_vector_b_batch(X / S) * S
    f.set_precision("mixed")
    mixed = f.calculate_vector_b(X[0] / S) * S
    f.close(), d.close()
    assert "m2l_product" in ran and "class_axial" in ran and "m2l_product" not in ref_ran
    err = lambda a, b, x: np.linalg.norm(a - b) / np.linalg.norm(b - x)
    e = [err(got, ref, X[0])] + [err(batch[r], ref_batch[r], X[r]) for r in range(3)]
    print(f"side {side}: {max(e):.1e}, mixed {err(mixed, got, X[0]):.1e}")
    assert max(e) < 1e-11 and err(mixed, got, X[0]) < 2e-5


@pytest.mark.parametrize("side,d0", [(180.0, 5.2), (190.0, 5.4)])
def test_most_degrees_of_the_small_kernel_and_one_more(side, d0):
    """32 and 33 last degrees for offsets of two boxes (test_host_enqueue.py pins which kernel
    shifts them): one and three right-hand sides against the class products of all degrees."""
    rng = np.random.default_rng(int(side))
    n = 260
    pos = rng.uniform(0.0, side, (n, 3))
    lmax = rng.integers(1, 5, n).astype(np.int32)
    args = (pos, 0.9 * lmax, 1.4 + 0.01j, 1.0)
    f = MultiSphereSolver(*args, lmax=lmax, use_fmm=True, leaf_size=32, fmm_d0=d0)
    d = MultiSphereSolver(*args, lmax=lmax, use_fmm=True, leaf_size=32, fmm_d0=d0, workspace_mb=4)
    S, mask = snm_flat(f.n_global, lmax)
    X = np.stack([(rng.standard_normal(f.n) + 1j * rng.standard_normal(f.n)) * mask for _ in range(3)])
    for batch in (X[:1], X):
        got, ref = f.calculate_vector_b_batch(batch / S) * S, d.calculate_vector_b_batch(batch / S) * S
        e = max(np.linalg.norm(got[r] - ref[r]) / np.linalg.norm(ref[r] - batch[r]) for r in range(len(batch)))
        print(f"side {side}, {len(batch)} right-hand sides: {e:.1e}")
        assert e < 1e-11
    f.close(), d.close()


def test_two_levels_against_the_direct_product():
    """Last degrees on two levels (nine spheres a box of the upper one) against all pairs, within the truncation of the
    boxes' expansions (d0 = 6; 1e-7 as for the other comparisons with the direct product)."""
    side, n = 270.0, 600
    rng = np.random.default_rng(270)
    i = np.arange(n)
    pos = (np.stack([i // 81, i // 9 % 9, i % 9], 1) + 0.5 + rng.uniform(-0.25, 0.25, (n, 3))) * side / 9
    lmax = rng.integers(1, 5, n).astype(np.int32)
    args = (pos, 0.9 * lmax, 1.4 + 0.01j, 1.0)
    f = MultiSphereSolver(*args, lmax=lmax, use_fmm=True, leaf_size=8)
    d = MultiSphereSolver(*args, lmax=lmax)
    S, mask = snm_flat(f.n_global, lmax)
    x = (rng.standard_normal(f.n) + 1j * rng.standard_normal(f.n)) * mask
    f.profile(True)
    got, ref = f.calculate_vector_b(x / S) * S, d.calculate_vector_b(x / S) * S
    ran = f.profile_read()
    levels = f.fmm_stats()[1]
    f.close(), d.close()
    e = np.linalg.norm(got - ref) / np.linalg.norm(ref - x)
    print(f"levels {levels}: {e:.1e}")
    assert len(levels) == 2 and "m2l_product" in ran and e < 1e-7
