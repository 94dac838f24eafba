"""M2L in the plane-wave basis: dense boxes on one and two levels, a sparse tree, both signs of
the translation vector, several right-hand sides at once and in groups that the workspace
forces, kept and regenerated tables, and one chunk of rows against many.  The spheres fill
their boxes, so offsets of every length occur, and at these orders the nearest ones leave
terms to the class products.

Reference: the class products (rotation, coaxial shift, rotation back) of the same tree and
box orders, which a workspace too small for the plane-wave samples falls back to: the same
truncated operator.  Both round at 1.1e-16 per term; the coaxial tables carry terms grown up
to 1e3 times within one of their bands and sums of up to 2 L = 300 terms, so 1e3 * 1.1e-16 *
sqrt(300) = 2e-12 of the translated part, and 1e-11 bounds the two.  Chunking and right-hand
sides change at most the order of sums: 1e-13."""
import numpy as np
import pytest

from helpers import snm_flat
from itofoggysim_amd import MultiSphereSolver

pytestmark = pytest.mark.gpu


def _spheres(n, side, seed, keep=lambda p: np.ones(len(p), bool)):
    rng = np.random.default_rng(seed)
    pos = rng.uniform(0.0, side, (4 * n, 3))
    pos = pos[keep(pos)][:n]
    return pos, rng.integers(1, 5, len(pos)).astype(np.int32)


CASES = {
    "one level": (300, 160.0, None, 8, {}),
    "two levels": (2500, 330.0, None, 16, {}),
    "sparse": (220, 190.0, lambda p: (p[:, 0] + p[:, 1] > 110.0), 4, {}),
    "reference sign": (300, 160.0, None, 8, dict(d_convention="reference")),
    "regenerated": (300, 160.0, None, 8, dict(cache_mb=-1)),
    "many chunks": (300, 160.0, None, 8, dict(workspace_mb=48)),
    "many chunks, regenerated": (300, 160.0, None, 8, dict(workspace_mb=48, cache_mb=-1)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_plane_wave_m2l_vs_class_products(name):
    n, side, keep, leaf, kw = CASES[name]
    pos, lmax = _spheres(n, side, 11 + n) if keep is None else _spheres(n, side, 11 + n, keep)
    n = len(pos)
    args = (pos, 0.9 * lmax, 1.4 + 0.01j, 1.0)
    conv = {k: v for k, v in kw.items() if k == "d_convention"}
    f = MultiSphereSolver(*args, lmax=lmax, use_fmm=True, leaf_size=leaf, fmm_d0=6.0, **kw)
    d = MultiSphereSolver(*args, lmax=lmax, use_fmm=True, leaf_size=leaf, fmm_d0=6.0, workspace_mb=4, **conv)
    S, mask = snm_flat(f.n_global, lmax)
    rng = np.random.default_rng(5)
    X = np.stack([(rng.standard_normal(f.n) + 1j * rng.standard_normal(f.n)) * mask for _ in range(3)])
    f.profile(True)
    b = [f.calculate_vector_b(x / S) * S for x in X]
    ran = f.profile_read()
    f.profile(False)
    both = f.calculate_vector_b_batch(X / S) * S
    again = f.calculate_vector_b(X[0] / S) * S
    d.profile(True)
    ref = [d.calculate_vector_b(x / S) * S for x in X]
    assert "m2l_product" not in d.profile_read()
    counts, levels = f.fmm_stats()
    f.close()
    d.close()
    assert "m2l_product" in ran, ran.keys()
    if name == "two levels":  # five spheres a leaf box: P2M and L2P by samples too
        assert "p2m_samples" in ran and "l2p_samples" in ran
    assert np.array_equal(again, b[0])
    for r in range(3):
        den = np.linalg.norm(ref[r] - X[r])
        e = np.linalg.norm(b[r] - ref[r]) / den
        eb = np.linalg.norm(both[r] - b[r]) / den
        print(name, levels, counts, f"vs class products {e:.2e}, batched vs single {eb:.2e}, synth launches",
              ran["m2l_synth"][1])
        assert e < 1e-11 and eb < 1e-13
