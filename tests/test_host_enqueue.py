"""What the library enqueues, on a runtime that records calls (host_runtime.py)."""
import pytest

import host_runtime


@pytest.fixture(scope="module")
def so(tmp_path_factory):
    return host_runtime.build(tmp_path_factory.mktemp("host_runtime"))


@pytest.mark.parametrize("args", ["12, 40.0, 1, 9", "400, 160.0, 1, 9, use_fmm=True, leaf_size=32"])
def test_creation_waits_for_its_kernels(so, args):
    """ifs_create's kernels run on the context's own stream, which orders nothing against the
    stream a caller sets next: none may be outstanding when it returns."""
    n, side, lo, hi, *kw = args.split(", ")
    host_runtime.run(so, f"""
s = solver(*spheres({n}, {side}, {lo}, {hi}), {", ".join(kw)})
seen = fake.calls()
own = {{c[2] for c in launches(seen)}}
assert len(own) == 1 and len(launches(seen)) > 1, seen
stream = own.pop()
last = max(i for i, c in enumerate(seen) if c[0] == "launch")
assert ["sync", stream] in seen[last:], seen[last:]
""")


WATCH = """
pointers = [("k_pair_fwdI", 9, 0), ("k_pair_axialI", 8, 0), ("k_pair_axialI", 10, 0), ("k_pair_backI", 7, 0),
            ("k_pair_backI", 9, 0), ("k_class_rot_fwd", 5, 0), ("k_class_rot_fwd", 6, 0), ("k_leaf_rows", 5, 0)]
pointers += [("k_pw_fft", 0, 144 + 8 * i) for i in range(5)]
for name, arg, offset in pointers:
    fake.fake_watch(name.encode(), arg, offset)
def behind(seen):
    out = {}
    for c in seen:
        if c[0] == "arg":
            key = tuple(c[1:4])
            out[key] = min(out.get(key, 1 << 62), int(c[4]))
    return out
"""


@pytest.mark.parametrize("args", ["12, 40.0, 1, 9", "400, 160.0, 1, 9, use_fmm=True, leaf_size=32"])
def test_a_failed_allocation_leaves_the_context_usable(so, args):
    """A batched product that runs out of memory at any of its allocations returns an error; the
    single product after it and the batched one, once there is memory again, find every
    workspace in place and as large as their plan needs."""
    n, side, lo, hi, *kw = args.split(", ")
    host_runtime.run(so, WATCH + f"""
import numpy as np
from itofoggysim_amd._lib import IfsError
def make():
    return solver(*spheres({n}, {side}, {lo}, {hi}), {", ".join(kw)})
s = make()
x = np.zeros((3, s.n), complex)
fake.calls()
s.calculate_vector_b(x[0])
single = behind(fake.calls())
before = fake.fake_allocs()
s.calculate_vector_b_batch(x)
batch = behind(fake.calls())
count = fake.fake_allocs() - before
assert single and batch and min(single.values()) > 0 and count > 4
s.close()
for granted in range(count):
    s = make()
    s.calculate_vector_b(x[0])
    fake.fake_fail_after(granted)
    try:
        s.calculate_vector_b_batch(x)
        failed = False
    except IfsError as e:
        failed = e.code == -2
    fake.fake_fail_after(-1)
    assert failed, granted
    for call, want in ((lambda: s.calculate_vector_b(x[0]), single), (lambda: s.calculate_vector_b_batch(x), batch)):
        fake.calls()
        call()
        got = behind(fake.calls())
        assert got.keys() == want.keys()
        assert all(got[k] >= want[k] for k in want if "pair" in k[0]), (granted, got, want)
        assert min(got.values()) > 0, (granted, got)
    s.close()
""")


@pytest.mark.parametrize("kw", ["", ", workspace_mb=4"])
def test_a_new_cut_of_box_translations_waits_for_the_old_one(so, kw):
    """Products with another number of right-hand sides replace the lists that the kernels of the
    product before them may still read: no list is written while a launch is outstanding."""
    host_runtime.run(so, f"""
s = solver(*spheres(400, 160.0, 1, 9), use_fmm=True, leaf_size=32{kw})
x, b = (ctypes.create_string_buffer(16 * 3 * s.n) for _ in range(2))
x, b = ctypes.addressof(x), ctypes.addressof(b)
replaced = 0
fake.calls()
for nrhs in (1, 3, 1, 3):
    s.calculate_vector_b_batch_device(x, b, nrhs)
outstanding = False
for c in fake.calls():
    if c[0] == "launch":
        outstanding = True
    elif c[0] == "sync":
        outstanding = False
    elif c[0] == "copy":
        replaced += 1
        assert not outstanding, c
assert replaced > 10
""")


@pytest.mark.parametrize("kw", ["", "workspace_mb=1", "workspace_mb=1, cache_mb=-1"])
def test_direct_products_of_any_number_of_right_hand_sides_only_enqueue(so, kw):
    """A direct plan serves every number of right-hand sides: once the vectors of the largest
    number have their room, products neither wait nor copy nor allocate, a caller's own capture of
    a batched one holds, and a captured single product is replayed beside batched ones."""
    host_runtime.run(so, f"""
s = solver(*spheres(40, 60.0, 1, 9), {kw})
x, b = (ctypes.create_string_buffer(16 * 5 * s.n) for _ in range(2))
x, b = ctypes.addressof(x), ctypes.addressof(b)
s.calculate_vector_b_batch_device(x, b, 5)
fake.calls()
for nrhs in (1, 3, 5, 2, 1):
    s.calculate_vector_b_batch_device(x, b, nrhs)
seen = fake.calls()
assert len(launches(seen, "k_finalize")) == 5 and len(launches(seen)) == len(seen), seen
stream = ctypes.c_void_p()
fake.hipStreamCreate(ctypes.byref(stream))
s.set_stream(stream.value)
graph = ctypes.c_void_p()
for nrhs in (1, 4):
    assert fake.hipStreamBeginCapture(stream, 1) == 0
    s.calculate_vector_b_batch_device(x, b, nrhs)
    assert fake.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
for _ in range(2):
    s.calculate_vector_b_graph_device(x, b)
fake.calls()
for _ in range(3):
    s.calculate_vector_b_graph_device(x, b)
    s.calculate_vector_b_batch_device(x, b, 3)
seen = fake.calls()
assert len([c for c in seen if c[0] == "graph"]) == 3
assert not [c for c in seen if c[0] not in ("graph", "launch")], seen
""")


def test_groups_of_right_hand_sides_share_one_plan(so):
    """Three right-hand sides in a workspace that holds the samples of two at once: the groups of
    two and one run on one plan, so repeated products neither wait nor copy, and a capture of one
    holds."""
    host_runtime.run(so, """
s = solver(*spheres(400, 160.0, 1, 9), use_fmm=True, leaf_size=32, workspace_mb=64)
x, b = (ctypes.create_string_buffer(16 * 3 * s.n) for _ in range(2))
x, b = ctypes.addressof(x), ctypes.addressof(b)
s.calculate_vector_b_batch_device(x, b, 3)
fake.calls()
s.calculate_vector_b_batch_device(x, b, 3)
seen = fake.calls()
assert len(launches(seen, "k_pw_unpack")) == 4  # leaf samples and box translations of two groups
assert not [c for c in seen if c[0] != "launch"], [c for c in seen if c[0] != "launch"]
stream, graph = ctypes.c_void_p(), ctypes.c_void_p()
fake.hipStreamCreate(ctypes.byref(stream))
s.set_stream(stream.value)
assert fake.hipStreamBeginCapture(stream, 1) == 0
s.calculate_vector_b_batch_device(x, b, 3)
assert fake.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
""")


def test_graph_products_between_batched_ones_of_a_tree(so):
    """An MLFMM context cuts its lists anew when the number of right-hand sides changes: not inside
    the capture of a graph product, where waiting and copying break the capture, and a graph whose
    lists are the ones it was captured with is replayed."""
    host_runtime.run(so, """
for kw in ({}, dict(workspace_mb=4)):
    s = solver(*spheres(400, 160.0, 1, 9), use_fmm=True, leaf_size=32, **kw)
    x, b = (ctypes.create_string_buffer(16 * 3 * s.n) for _ in range(2))
    x, b = ctypes.addressof(x), ctypes.addressof(b)
    s.calculate_vector_b_batch_device(x, b, 3)
    fake.calls()
    for _ in range(2):
        for _ in range(3):
            s.calculate_vector_b_graph_device(x, b)
        s.calculate_vector_b_batch_device(x, b, 3)
    s.calculate_vector_b_graph_device(x, b)
    seen = fake.calls()
    inside = False
    for c in seen:
        if c[0] == "capture":
            inside = True
        elif c[0] == "captured":
            inside = False
        assert not inside or c[0] in ("capture", "launch"), c
    assert len([c for c in seen if c[0] == "captured"]) == 1, seen
    assert len([c for c in seen if c[0] == "graph"]) == 6
    s.close()
""")


def test_tables_in_fp32_only_for_contexts_that_run_mixed(so):
    """FP64 contexts hold no FP32 copy of the plane-wave tables; the first mixed product brings one,
    once, where the cache budget has room, and a captured one that comes first runs on the FP64 tables."""
    host_runtime.run(so, """
make = lambda **kw: solver(*spheres(400, 160.0, 1, 9), use_fmm=True, leaf_size=32, **kw)
x, b = (ctypes.create_string_buffer(16 << 20) for _ in range(2))
x, b = ctypes.addressof(x), ctypes.addressof(b)
def held(s):
    for _ in range(2):
        s.calculate_vector_b_device(x, b)
    return fake.fake_live_bytes()
s = make()
fp64 = held(s)
s.set_precision("mixed")
late = held(s) - fp64
s.calculate_vector_b_device(x, b)
fake.calls()
s.calculate_vector_b_device(x, b)
seen = fake.calls()
assert len(launches(seen)) == len(seen) and not launches(seen, "k_pw_ttable"), seen
s.close()
s = make(precision="mixed")
assert held(s) - fp64 == late > 0
s.close()
s = make()
stream, graph = ctypes.c_void_p(), ctypes.c_void_p()
fake.hipStreamCreate(ctypes.byref(stream))
s.set_stream(stream.value)
s.set_class_tiles(64, 64, False)
s.calculate_vector_b_device(x, b)
s.set_precision("mixed")
fake.calls()
assert fake.hipStreamBeginCapture(stream, 1) == 0
s.calculate_vector_b_device(x, b)
assert fake.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
assert launches(fake.calls(), "k_pw_m2lI15HIP_vector_typeIdLj2EE")
s.close()
# the smallest budget that holds every table of FP64 products: they stay when mixed ones follow
def warm(s):
    held(s)
    fake.calls()
    s.calculate_vector_b_device(x, b)
    return len(launches(fake.calls()))
s = make()
all_kept = warm(s)
mb = 1
while True:
    s = make(cache_mb=mb)
    if warm(s) == all_kept:
        break
    mb += 1
    s.close()
assert mb < fp64 >> 20
s.set_precision("mixed")
assert warm(s) == all_kept
s.set_precision("fp64")
assert warm(s) == all_kept
""")


@pytest.mark.parametrize("big,side", [(520, 200.0), (420, 3140.0)])
def test_samples_of_leaf_boxes_only_where_local_memory_holds_them(so, big, side):
    """One sphere of a very high order (row sums of 64 KiB a pair of spheres), and high box and sphere
    orders together (a quarter of a row's azimuths): no launch beyond the 64 KiB of a block."""
    host_runtime.run(so, f"""
import numpy as np
pos, lmax = spheres(12, {side}, 1, 4)
pos *= 0.3
pos[-1] = {side}
lmax[3] = {big}
s = solver(pos, lmax, use_fmm=True, leaf_size=12)
x, b = (ctypes.create_string_buffer(16 * s.n) for _ in range(2))
s.calculate_vector_b_device(ctypes.addressof(x), ctypes.addressof(b))
seen = fake.calls()
assert not [c for c in seen if c[0] == "refused"], [c for c in seen if c[0] == "refused"]
assert not launches(seen, "k_leaf")
""")


@pytest.mark.parametrize("side,d0,blocks", [(180.0, 5.2, False), (190.0, 5.4, True)])
def test_last_degrees_by_the_thread_kernel_up_to_32(so, side, d0, blocks):
    """What the plane waves leave of near offsets is shifted by one thread a translation up to 32 degrees
    (offsets of two boxes: 32 and 33 in these trees) and by 64-row blocks beyond."""
    host_runtime.run(so, f"""
import numpy as np
rng = np.random.default_rng(int({side}))
pos = rng.uniform(0.0, {side}, (260, 3))
lmax = rng.integers(1, 5, 260).astype(np.int32)
s = solver(pos, lmax, use_fmm=True, leaf_size=32, fmm_d0={d0})
x, b = (ctypes.create_string_buffer(16 * s.n) for _ in range(2))
fake.calls()
s.profile(True)
s.calculate_vector_b_device(ctypes.addressof(x), ctypes.addressof(b))
seen = fake.calls()
ran = s.profile_read()  # one level, no whole offset: only 33 degrees run as class products by blocks
assert "class_axial_rem" in ran and ("class_axial" in ran) == {blocks}
assert launches(seen, "k_class_axial_remI") and launches(seen, "k_pw_m2l")
assert bool(launches(seen, "k_class_axialI")) == {blocks}, [c[1] for c in launches(seen, "k_class")]
""")


@pytest.mark.parametrize("gen,n,ndir,fmm,precision,budget", [
    ("uniform", 20, 1, False, "fp64", 200.0), ("uniform", 180, 2, False, "fp64", 8.0),
    ("uniform", 250, 1, True, "fp64", 200.0), ("uniform", 500, 8, True, "fp64", 200.0),
    ("uniform", 2500, 1, True, "mixed", 200.0), ("lognormal", 200, 2, True, "mixed", 200.0)])
def test_a_served_request_stays_in_its_plan_and_keeps_its_tables(so, gen, n, ndir, fmm, precision, budget):
    """A context made with the limits that the server's plan gives it: what it allocates for products
    of all directions is what the plan holds beside the Krylov basis, which in turn is no more than
    twice that (and 256 MiB), and the second product generates no table.  180 spheres in a share of 2
    GiB: the tables of all pairs are 75 MiB."""
    host_runtime.run(so, f"""
import numpy as np
from itofoggysim_amd import MultiSphereSolver, config_cluster, make_cluster, plan_request
c = make_cluster({n}, ("uniform", 0.3, 1.0), side=10.0 * ({n} / 20.0) ** (1.0 / 3.0), seed={n}) \
    if {gen!r} == "uniform" else config_cluster(2, n={n})
p = plan_request(c["centres"], c["radii"], c["k"], {ndir}, lmax=c["lmax"], use_fmm={fmm}, precision={precision!r},
                 hbm_budget_gb={budget}, slots=4)
fake.fake_set_free(250 << 30)
s = MultiSphereSolver(c["centres"], c["radii"], 1.33, c["k"], lmax=c["lmax"], use_fmm={fmm}, leaf_size=32,
                      precision={precision!r}, workspace_mb=p["workspace_mb"], cache_mb=p["cache_mb"])
x = ctypes.create_string_buffer(64)
for _ in range(2):
    fake.calls()
    s.calculate_vector_b_batch_device(ctypes.addressof(x), ctypes.addressof(x), {ndir})
made = [k[1] for k in launches(fake.calls()) if any(t in k[1] for t in ("table", "k_gen", "k_gq"))]
live = fake.fake_live_bytes()
basis = 16.0 * s.n * 31 * {ndir}
print({n}, {ndir}, "live", live / 2 ** 20, "MiB, plan", (p["total"] - basis) / 2 ** 20, made)
assert not made and live <= p["total"] - basis
assert p["total"] - p["vectors"] <= 2.0 * live + (256 << 20)
""")


def test_profile_counts_the_flops_of_every_product(so):
    """Each kernel group of an MLFMM product that multiplies reports its algorithmic flops, in proportion to
    the right-hand sides and whatever the chunks; the sampled translations 16 flops per sample of the
    grid and translation."""
    host_runtime.run(so, """
import numpy as np
def flops(nrhs, **kw):
    s = solver(*spheres(400, 160.0, 1, 9), use_fmm=True, leaf_size=32, **kw)
    x = ctypes.create_string_buffer(64)
    s.profile(True)
    s.calculate_vector_b_batch_device(ctypes.addressof(x), ctypes.addressof(x), nrhs)
    f = {k: v[2] for k, v in s.profile_read().items()}
    (L,), m2l = s.fmm_stats()[1].values(), s.fmm_stats()[0]["M2L"]
    total = s.matvec_cost()[0]
    s.close()
    return f, L, m2l, total
f, L, m2l, total = flops(1)
names = ["m2l_synth", "m2l_fft", "m2l_product", "m2l_anal", "p2m_samples", "p2m_box", "l2p_box", "l2p_samples",
         "l2p_sum", "p2p_rot_fwd", "p2p_axial", "p2p_rot_back", "class_rot_fwd", "class_axial", "class_axial_rem",
         "class_rot_back"]
assert all(f[k] > 0.0 for k in names), f
samples = f["m2l_product"] / (16.0 * m2l)  # few offsets are class products as a whole
assert 2 * (L + 1) * L < samples < 2 * (L + 1) * (4 * L + 100), (samples, L)
assert f["m2l_synth"] == f["m2l_anal"] and f["m2l_synth"] + f["m2l_fft"] + f["m2l_anal"] + f["m2l_product"] < total
for kw in ({}, dict(workspace_mb=64)):
    g = flops(3, **kw)[0]
    for k in names:
        if not (kw and k.startswith("l2p_box")):  # boxes are sampled again for each group of spheres
            assert abs(g[k] - 3.0 * f[k]) < 1e-12 * g[k], (k, kw, f[k], g[k])
""")


@pytest.mark.parametrize("args", ["12, 40.0, 1, 9", "400, 160.0, 1, 9, use_fmm=True, leaf_size=32",
                                  "400, 160.0, 1, 9, use_fmm=True, leaf_size=32, workspace_mb=4",
                                  "3, 200.0, 60, 66"])
def test_tables_of_a_captured_first_product_stay_to_be_made(so, args):
    """A caller's capture may hold a context's first product: its table kernels are recorded, not run, so an
    eager product beside the graph makes the tables itself; those after it find them."""
    n, side, lo, hi, *kw = args.split(", ")
    host_runtime.run(so, f"""
s = solver(*spheres({n}, {side}, {lo}, {hi}), {", ".join(kw)})
x = ctypes.create_string_buffer(64)
stream, graph = ctypes.c_void_p(), ctypes.c_void_p()
fake.hipStreamCreate(ctypes.byref(stream))
s.set_stream(stream.value)
def tables():
    fake.calls()
    s.calculate_vector_b_device(ctypes.addressof(x), ctypes.addressof(x))
    return [c[1] for c in launches(fake.calls()) if any(t in c[1] for t in ("table", "k_gen", "k_gq"))]
assert fake.hipStreamBeginCapture(stream, 1) == 0
captured = tables()
assert fake.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
assert captured and set(tables()) == set(captured)
assert not tables()
""")
