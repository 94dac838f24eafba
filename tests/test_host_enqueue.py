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
