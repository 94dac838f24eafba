"""Direct products whose last kernel adds the partial sums of each sphere (all pairs in one
chunk of the workspace) against the separate reduction of several chunks: a sphere alone in
its cluster (no sums), clusters with few and with many pairs per sphere (one and several
partial sums), rows without a target (the rows of all spheres in chunks, those of the others
replaced), one and three right-hand sides.  Only the grouping of
at most 40 terms of a sum may differ: 1e-14 of the largest entry."""
import numpy as np
import pytest

from itofoggysim_amd import ClusterBatch, MultiSphereSolver

pytestmark = pytest.mark.gpu


def _cluster(n, rng):
    lmax = rng.integers(2, 8, n).astype(np.int32)
    g = np.arange(n)
    pos = (np.stack([g // 16, g // 4 % 4, g % 4], 1) + rng.uniform(-0.2, 0.2, (n, 3))) * 8.0
    return dict(centres=pos, radii=0.5 * lmax, m_rel=1.4 + 0.01j, lmax=lmax)


@pytest.mark.parametrize("name", ["clusters", "zeroed rows"])
def test_partial_sums_equal_reduction(name):
    rng = np.random.default_rng(3)
    if name == "clusters":
        cl = [_cluster(n, rng) for n in (1, 2, 5, 40)]
        make = lambda **kw: ClusterBatch(cl, 1.0, **kw)
    else:
        c = _cluster(40, rng)
        make = lambda z=False, **kw: MultiSphereSolver(c["centres"], c["radii"], c["m_rel"], 1.0, lmax=c["lmax"],
                                                       ref_row_zeroing=z, **kw)
    a = make() if name == "clusters" else make(z=True)
    b = make(workspace_mb=1)
    X = rng.standard_normal((3, a.n)) + 1j * rng.standard_normal((3, a.n))
    for x in (X[:1], X):
        got, ref = a.calculate_vector_b_batch(x), b.calculate_vector_b_batch(x)
        if name == "zeroed rows":  # b = x where a sphere is no target
            off = np.repeat(c["lmax"] < c["lmax"].max(), a.n // 40)
            ref = np.where(off, x, ref)
            assert np.array_equal(got[:, off], x[:, off])
        for r in range(len(x)):
            assert np.max(np.abs(got[r] - ref[r])) <= 1e-14 * np.max(np.abs(ref[r]))
    a.profile(True), b.profile(True)
    assert np.array_equal(a.calculate_vector_b(X[0]), got[0])
    b.calculate_vector_b(X[0])
    assert "zero" not in a.profile_read() and "zero" in b.profile_read()
    a.close(), b.close()
