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
