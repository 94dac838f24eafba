"""Products of changing numbers of right-hand sides, and on a stream set directly after creation:

  * single products replayed as a graph between batched ones of two and three right-hand sides;
    direct plans of the pair kernels, a direct plan whose largest sphere (order 66) is beyond
    them, and an MLFMM whose workspace holds two right-hand sides at once, so that three run in
    groups of two and one;
  * the first product of a context on a caller's own stream;
  * a context's first product inside a caller's capture, then an eager one, then the captured one.

A replay runs the captured launches on the same buffers: equal bits.  Direct batched products
take the same sums per right-hand side: equal bits.  In the MLFMM the number of right-hand sides
changes how rows are cut into chunks, so the order of sums of at most some hundred terms: 1e-13 of
the translated part, as in the box translations' own test.  The order-66 sphere is compared with the
oracle per target sphere at 1e-10, the bound of the other tests of high orders."""
import ctypes

import numpy as np
import pytest

from helpers import Hip, per_sphere_rel, snm_flat
from itofoggysim_amd import MultiSphereSolver

pytestmark = pytest.mark.gpu


def _spheres(n, side, lo, hi, seed):
    rng = np.random.default_rng(seed)
    g = int(np.ceil(n ** (1.0 / 3.0)))
    i = np.arange(n)
    pos = (np.stack([i // g ** 2, i // g % g, i % g], 1) + 0.5 + rng.uniform(-0.25, 0.25, (n, 3))) * side / g
    return pos, rng.integers(lo, hi + 1, n).astype(np.int32)


def _make(name):
    if name == "order 66":
        pos, lmax = np.array([[0.0, 0.0, 0.0], [60.0, 25.0, 30.0], [-20.0, 70.0, -55.0]]), np.array([66, 9, 4], np.int32)
        return pos, lmax, MultiSphereSolver(pos, 0.75 * lmax, 1.4 + 0.01j, 1.0, lmax=lmax)
    if name == "direct":
        pos, lmax = _spheres(40, 60.0, 1, 9, 3)
        return pos, lmax, MultiSphereSolver(pos, 0.75 * lmax, 1.4 + 0.01j, 1.0, lmax=lmax)
    pos, lmax = _spheres(400, 160.0, 1, 9, 4)
    return pos, lmax, MultiSphereSolver(pos, 0.75 * lmax, 1.4 + 0.01j, 1.0, lmax=lmax, use_fmm=True, leaf_size=32,
                                        workspace_mb=64)


@pytest.mark.parametrize("name", ["direct", "order 66", "MLFMM"])
def test_single_graph_replays_between_batched_products(oracle, name):
    pos, lmax, s = _make(name)
    S, mask = snm_flat(s.n_global, lmax)
    rng = np.random.default_rng(8)
    X = np.stack([(rng.standard_normal(s.n) + 1j * rng.standard_normal(s.n)) * mask for _ in range(3)])
    single = np.stack([s.calculate_vector_b(x / S) for x in X])
    hip = Hip()
    try:
        x, b = hip.upload(X / S), hip.upload(np.zeros_like(X))
        for count in (1, 1, 1, 3, 1, 2, 1, 1, 3):
            if count == 1:
                s.calculate_vector_b_graph_device(x.value, b.value)
            else:
                s.calculate_vector_b_batch_device(x.value, b.value, count)
            hip.sync(s.stream())
            got = hip.download(b, X)[:count]
            for r in range(count):
                if name == "MLFMM" and count > 1:
                    e = np.linalg.norm((got[r] - single[r]) * S) / np.linalg.norm(single[r] * S - X[r])
                    assert e < 1e-13, (count, r, e)
                else:
                    assert np.array_equal(got[r], single[r]), (count, r)
        if name == "order 66":
            an, bn = s.mie_coefficients()
            for r in range(3):
                ref = oracle.matvec_direct(-pos, lmax, s.n_global, an, bn, 1.0, X[r] / S) * S
                e = per_sphere_rel(single[r] * S, ref, X[r], len(lmax), s.n_global)
                print("order 66, per target", e)
                assert e.max() < 1e-10
    finally:
        hip.free_all()
        s.close()


@pytest.mark.parametrize("name", ["direct", "MLFMM"])
def test_first_product_on_a_stream_set_after_creation(name):
    hip = Hip()
    stream = ctypes.c_void_p()
    assert hip.rt.hipStreamCreateWithFlags(ctypes.byref(stream), 1) == 0
    out = []
    rng = np.random.default_rng(9)
    v = None
    for early in (True, False):
        _, lmax, s = _make(name)
        if early:
            s.set_stream(stream.value)
        if v is None:
            S, mask = snm_flat(s.n_global, lmax)
            v = (rng.standard_normal(s.n) + 1j * rng.standard_normal(s.n)) * mask / S
        x, b = hip.upload(v), hip.upload(np.zeros_like(v))
        s.calculate_vector_b_device(x.value, b.value)
        hip.sync(s.stream())
        out.append(hip.download(b, v))
        s.close()
    hip.free_all()
    assert hip.rt.hipStreamDestroy(stream) == 0
    assert np.array_equal(out[0], out[1]) and np.isfinite(out[0]).all()


@pytest.mark.parametrize("name", ["direct", "order 66", "MLFMM"])
def test_first_product_in_a_callers_capture(name):
    hip = Hip()
    rt, stream = hip.rt, ctypes.c_void_p()
    assert rt.hipStreamCreateWithFlags(ctypes.byref(stream), 1) == 0
    _, lmax, s = _make(name)
    S, mask = snm_flat(s.n_global, lmax)
    rng = np.random.default_rng(10)
    v = (rng.standard_normal(s.n) + 1j * rng.standard_normal(s.n)) * mask / S
    s.set_class_tiles(64, 64, False)
    want = s.calculate_vector_b(v)
    s.close()
    _, _, s = _make(name)
    s.set_class_tiles(64, 64, False)
    s.set_stream(stream.value)
    x, b, g = hip.upload(v), hip.upload(np.zeros_like(v)), hip.upload(np.zeros_like(v))
    graph, run = ctypes.c_void_p(), ctypes.c_void_p()
    assert rt.hipStreamBeginCapture(stream, 1) == 0
    s.calculate_vector_b_device(x.value, g.value)
    assert rt.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    s.calculate_vector_b_device(x.value, b.value)
    hip.sync(stream)
    assert np.array_equal(hip.download(b, v), want)
    assert rt.hipGraphInstantiate(ctypes.byref(run), graph, None, None, 0) == 0
    for _ in range(2):
        assert rt.hipGraphLaunch(run, stream) == 0
        s.calculate_vector_b_device(x.value, b.value)
        hip.sync(stream)
        assert np.array_equal(hip.download(g, v), want) and np.array_equal(hip.download(b, v), want)
    rt.hipGraphExecDestroy(run), rt.hipGraphDestroy(graph)
    s.close()
    hip.free_all()
    assert rt.hipStreamDestroy(stream) == 0
