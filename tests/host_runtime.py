"""The library's host code on a HIP runtime that records calls instead of making them
(host_runtime.cpp): what is enqueued on which stream, where the host waits, and what a
failed allocation leaves behind.  Runs in a process of its own, which loads the stand-in
before libifs.so; no GPU is used and no kernel runs."""
import ctypes
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def build(directory):
    """Compiles the stand-in into `directory`; its path."""
    so = os.path.join(str(directory), "libhost_runtime.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-o", so, os.path.join(HERE, "host_runtime.cpp")],
                   check=True)
    return so


def run(so, body):
    """Runs the Python source `body` beside the stand-in (`fake`, and this module's helpers);
    fails with its output if it fails."""
    code = f"import sys; sys.path[:0] = [{ROOT!r}, {HERE!r}]\nfrom host_runtime import *\nfake = load({so!r})\n" + body
    p = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stdout + p.stderr


def load(so):
    f = ctypes.CDLL(so, mode=ctypes.RTLD_GLOBAL)
    f.fake_log.restype = ctypes.c_char_p
    f.fake_live_bytes.restype = ctypes.c_longlong
    f.fake_allocs.restype = ctypes.c_long
    f.fake_fail_after.argtypes = [ctypes.c_long]
    f.fake_set_free.argtypes = [ctypes.c_size_t]
    f.fake_watch.argtypes = [ctypes.c_char_p, ctypes.c_int, ctypes.c_size_t]

    def calls(clear=True):
        out = [l.split() for l in f.fake_log().decode().splitlines()]
        if clear:
            f.fake_clear()
        return out

    f.calls = calls
    return f


def launches(calls, kernel=""):
    return [c for c in calls if c[0] == "launch" and kernel in c[1]]


def spheres(n, side, lo, hi, seed=1):
    """Jittered lattice of n spheres of orders lo..hi in a cube (centres, orders)."""
    import numpy as np
    rng = np.random.default_rng(seed)
    g = int(np.ceil(n ** (1.0 / 3.0)))
    i = np.arange(n)
    pos = (np.stack([i // g ** 2, i // g % g, i % g], 1) + 0.5 + rng.uniform(-0.25, 0.25, (n, 3))) * side / g
    pos[0], pos[-1] = 0.0, side
    return pos, rng.integers(lo, hi + 1, n).astype(np.int32)


def solver(pos, lmax, **kw):
    from itofoggysim_amd import MultiSphereSolver
    return MultiSphereSolver(pos, 0.8 * lmax, 1.4 + 0.01j, 1.0, lmax=lmax, **kw)
