"""P2M and L2P through samples of the leaf boxes' fields: spheres of orders 1 to 9 and one of
13 (every class of the order mod 4), none nearer than half a lattice spacing, in boxes that hold several, empty rows (spheres without a
target row), kept and regenerated tables, row chunks and sphere groups that a small
workspace forces, and three right-hand sides.

Reference: the translations one by one (rotation, coaxial quadrature, rotation back), which a
workspace too small for the samples falls back to, on the same tree; the box translations
fall back with them.  All factors have modulus one and the sums at most 200 terms, so the
two differ by the coaxial tables' 2e-12 (see the box translations' test): 1e-11 of the translated
part.  Chunks, groups and right-hand sides change at most the order of sums: 1e-13."""
import numpy as np
import pytest

from helpers import snm_flat
from itofoggysim_amd import MultiSphereSolver

pytestmark = pytest.mark.gpu

CASES = {
    "dense": (400, 160.0, 32, {}),
    "zeroed rows": (400, 160.0, 32, dict(ref_row_zeroing=True)),
    "regenerated": (400, 160.0, 32, dict(cache_mb=-1)),
    "chunks and groups": (400, 160.0, 32, dict(workspace_mb=48)),
    "chunks, regenerated": (400, 160.0, 32, dict(workspace_mb=48, cache_mb=-1)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_leaf_samples_vs_translations(name):
    n, side, leaf, kw = CASES[name]
    rng = np.random.default_rng(n)
    g = int(np.ceil(n ** (1.0 / 3.0))) + 1  # a jittered lattice: the nearest pairs do not outweigh the far field
    site = rng.permutation(g ** 3)[:n]
    pos = (np.stack([site // g ** 2, site // g % g, site % g], 1) + 0.5 + rng.uniform(-0.25, 0.25, (n, 3))) * side / g
    lmax = rng.integers(1, 10, n).astype(np.int32)
    lmax[7] = 13
    pos[np.argmax(pos.sum(1))] = side  # a corner of the tree
    args = (pos, 0.8 * lmax, 1.4 + 0.01j, 1.0)
    ref_kw = {k: v for k, v in kw.items() if k == "ref_row_zeroing"}
    f = MultiSphereSolver(*args, lmax=lmax, use_fmm=True, leaf_size=leaf, **kw)
    d = MultiSphereSolver(*args, lmax=lmax, use_fmm=True, leaf_size=leaf, workspace_mb=4, **ref_kw)
    S, mask = snm_flat(f.n_global, lmax)
    X = np.stack([(rng.standard_normal(f.n) + 1j * rng.standard_normal(f.n)) * mask for _ in range(3)])
    f.profile(True)
    b = [f.calculate_vector_b(x / S) * S for x in X]
    ran = f.profile_read()
    f.profile(False)
    both = f.calculate_vector_b_batch(X / S) * S
    again = f.calculate_vector_b(X[0] / S) * S
    d.profile(True)
    ref = [d.calculate_vector_b(x / S) * S for x in X]
    ref_ran = d.profile_read()
    f.close()
    d.close()
    assert "p2m_samples" in ran and "l2p_samples" in ran and "p2m_samples" not in ref_ran
    assert np.array_equal(again, b[0])
    for r in range(3):
        den = np.linalg.norm(ref[r] - X[r])
        e = np.linalg.norm(b[r] - ref[r]) / den
        eb = np.linalg.norm(both[r] - b[r]) / den
        print(name, f"vs translations {e:.2e}, batched vs single {eb:.2e}, sample launches", ran["l2p_samples"][1])
        assert e < 1e-11 and eb < 1e-13


def test_leaf_samples_of_larger_spheres():
    """Orders 31, 32 and 40 among small spheres: up to 31 one pass of a block covers an order's sums
    over the azimuths, beyond it two do; against all pairs.  The large spheres stand alone near the
    middle of their boxes: one that reaches beyond its box reads back degrees at which |h1| has grown
    to 1e12, where the one-by-one translations differ from themselves by 5e-9 to 4e-7 (kept against
    regenerated tables).  Inside, no sphere reaches beyond degree 85 of the box's 139, so the
    truncation vanishes and the bound of the translations holds for the direct product too."""
    edge, rng = 110.0, np.random.default_rng(41)
    pos, lmax = [], []
    for b in range(64):
        mid = (np.array([b // 16, b // 4 % 4, b % 4]) + 0.5) * edge
        big = {0: 31, 22: 32, 63: 40}.get(b)
        for k in range(1 if big else 2):  # two small spheres on different sides of the middle
            off = rng.uniform(-5.0, 5.0, 3) if big else (2 * k - 1) * rng.uniform(10.0, 35.0, 3)
            pos.append(mid + off)
            lmax.append(big or rng.integers(1, 10))
    pos += [np.zeros(3), np.full(3, 4 * edge)]  # corners of the tree
    pos, lmax = np.array(pos), np.array(lmax + [1, 1], np.int32)
    n = len(pos)
    args = (pos, 0.8 * lmax, 1.4 + 0.01j, 1.0)
    f = MultiSphereSolver(*args, lmax=lmax, use_fmm=True, leaf_size=32)
    d = MultiSphereSolver(*args, lmax=lmax)
    S, mask = snm_flat(f.n_global, lmax)
    x = (rng.standard_normal(f.n) + 1j * rng.standard_normal(f.n)) * mask
    f.profile(True)
    got, ref = f.calculate_vector_b(x / S) * S, d.calculate_vector_b(x / S) * S
    ran = f.profile_read()
    f.close(), d.close()
    assert "l2p_samples" in ran
    got, ref, x = (v.reshape(n, -1) for v in (got, ref, x))
    for j in np.concatenate([np.flatnonzero(lmax > 30), [1, 50]]):
        e = np.linalg.norm(got[j] - ref[j]) / np.linalg.norm(ref[j] - x[j])
        print(f"order {lmax[j]}: {e:.2e}")
        assert e < 1e-11
    assert np.linalg.norm(got - ref) / np.linalg.norm(ref - x) < 1e-11
