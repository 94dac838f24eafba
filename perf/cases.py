"""Performance cases: what a program built on this framework has it do.

Five kinds of call, each through the package's public entry points:

  host    the GMRES callback on host arrays, b = (I + T A) x (``calculate_vector_b``): how a
          CPU solver with its own Krylov loop uses the library
  device  the same product on device vectors, direct or MLFMM, FP64 or mixed precision, one or
          several right-hand sides, eager or replayed as a HIP graph
  multi   one product over many independent clusters held in one context (``ClusterBatch``)
  solve   a whole GMRES solve for a plane wave (``solve``)
  far     the far field of a solved cluster on an angular grid (``far_field``)

Clusters come from the package's own generators: radii uniform in [0.3, 1] um at 20 spheres per
(10 um)^3 ("uniform"), or lognormal (median 1 um, sigma_g 1.5) at volume fraction 1e-3
("lognormal"), water index, wavelengths from 400 to 1550 nm.  The vectors are what a Krylov
loop hands to the product: coefficients of order one up to each sphere's size parameter that
fall off beyond it, in the flat layout.  Products are returned in the normalised basis
s_nm x_nm, in which such programs take their norms (flat entries span 1e+-80).
"""
import math

import numpy as np
import torch

from itofoggysim_amd import ClusterBatch, MultiSphereSolver, make_cluster
from itofoggysim_amd.cluster import lmax_rule

WATER = {0.55: complex(1.333, 1e-9), 1.55: complex(1.318, 1e-4)}


def listed():
    return [
        # the smallest request: a dozen spheres in the near infrared, the product replayed as a
        # graph inside a device-resident Krylov loop (latency and launches)
        dict(name="graph_12", kind="device", gen="uniform", n=12, wavelength=1.55, fmm=False, graph=True),
        # the 20-sphere benchmark cluster under a host GMRES: the callback with its copies
        dict(name="callback_20", kind="host", gen="uniform", n=20, wavelength=0.55, fmm=False),
        # an ordinary served request solved directly: all pairs of a ragged number of spheres
        dict(name="direct_151", kind="device", gen="uniform", n=151, wavelength=0.8, fmm=False, graph=False),
        # a batch of small clusters (parameter studies): 48 clusters of 5 to 40 spheres, one product
        dict(name="multi_48", kind="multi", gen="uniform", clusters=48, n_lo=5, n_hi=40, wavelength=0.55),
        # a whole request: GMRES to 1e-6 on a direct plan, right-hand side and solution on the host
        dict(name="solve_40", kind="solve", gen="uniform", n=40, wavelength=0.55, tol=1e-6, restart=30),
        # what follows a solve: the far field on the 181 x 36 angular grid
        dict(name="far_200", kind="far", gen="uniform", n=200, wavelength=0.55, ntheta=181, nphi=36),
        # MLFMM with small boxes: many spheres at a long wavelength (box orders 40 to 100)
        dict(name="mlfmm_3000_ir", kind="device", gen="uniform", n=3000, wavelength=1.55, fmm=True, mixed=False,
             nrhs=1, leaf=32),
        # the dense cloud at 550 nm: near field and box translations both count
        dict(name="mlfmm_2500", kind="device", gen="uniform", n=2500, wavelength=0.55, fmm=True, mixed=False,
             nrhs=1, leaf=32),
        # the dilute cloud of large droplets: box orders of several hundred dominate
        dict(name="mlfmm_droplets_333", kind="device", gen="lognormal", n=333, wavelength=0.55, fmm=True,
             mixed=False, nrhs=1, leaf=16),
        # the same kind of cloud in mixed precision, kept in 32 bits by the caller
        dict(name="mixed_droplets_200", kind="device", gen="lognormal", n=200, wavelength=0.55, fmm=True,
             mixed=True, nrhs=1, leaf=16),
        # four polarisations and directions of one cluster advanced in lock step
        dict(name="batch4_700", kind="device", gen="uniform", n=700, wavelength=0.55, fmm=True, mixed=False,
             nrhs=4, leaf=32),
    ]


def _between(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["graph", "host", "direct", "multi", "solve", "far", "mlfmm", "mlfmm", "droplets", "droplets",
                       "batch"])
    lam = round(rng.uniform(0.4, 1.55), 4)
    if kind == "graph":
        return dict(kind="device", gen="uniform", n=_between(rng, 10, 40), wavelength=round(rng.uniform(0.8, 1.55), 4),
                    fmm=False, graph=True)
    if kind == "host":
        return dict(kind="host", gen="uniform", n=_between(rng, 10, 80), wavelength=lam, fmm=False)
    if kind == "direct":
        return dict(kind="device", gen="uniform", n=_between(rng, 30, 200), wavelength=round(rng.uniform(0.6, 1.55), 4),
                    fmm=False, graph=False)
    if kind == "multi":
        return dict(kind="multi", gen="uniform", clusters=_between(rng, 8, 64), n_lo=5, n_hi=rng.randint(15, 40),
                    wavelength=round(rng.uniform(0.55, 1.55), 4))
    if kind == "solve":
        return dict(kind="solve", gen="uniform", n=_between(rng, 10, 60), wavelength=round(rng.uniform(0.5, 1.55), 4),
                    tol=1e-6, restart=30)
    if kind == "far":
        return dict(kind="far", gen="uniform", n=_between(rng, 20, 300), wavelength=round(rng.uniform(0.5, 1.55), 4),
                    ntheta=rng.randint(91, 181), nphi=rng.randint(1, 36))
    if kind == "mlfmm":
        return dict(kind="device", gen="uniform", n=_between(rng, 250, 2500), wavelength=round(rng.uniform(0.55, 1.55), 4),
                    fmm=True, mixed=False, nrhs=1, leaf=32)
    if kind == "droplets":
        return dict(kind="device", gen="lognormal", n=_between(rng, 60, 330), wavelength=round(rng.uniform(0.55, 1.1), 4),
                    fmm=True, mixed=rng.random() < 0.4, nrhs=1, leaf=rng.choice([16, 32]))
    return dict(kind="device", gen="uniform", n=_between(rng, 200, 700), wavelength=round(rng.uniform(0.55, 1.55), 4),
                fmm=True, mixed=False, nrhs=rng.randint(2, 4), leaf=32)


# -- inputs -------------------------------------------------------------------
def _index(lam):
    return WATER.get(lam, complex(1.3199 + 3500e-6 / lam ** 2, 1e-8))


def _cluster(case, seed, n=None):
    n = n or case["n"]
    if case["gen"] == "uniform":
        return make_cluster(n, ("uniform", 0.3, 1.0), side=10.0 * (n / 20.0) ** (1.0 / 3.0),
                            wavelength=case["wavelength"], m=_index(case["wavelength"]), seed=seed)
    return make_cluster(n, ("lognormal", 1.0, 1.5, 0.2, 3.0), volume_fraction=1e-3, wavelength=case["wavelength"],
                        m=_index(case["wavelength"]), seed=seed)


def _clusters(case, seed):
    if case["kind"] != "multi":
        return [_cluster(case, seed)]
    sizes = np.random.default_rng(case["clusters"]).integers(case["n_lo"], case["n_hi"] + 1, case["clusters"])
    return [_cluster(case, 1000 * seed + g, int(n)) for g, n in enumerate(sizes)]


def _degrees(N):
    n = np.repeat(np.arange(1, N + 1), 2 * np.arange(1, N + 1) + 1)
    return n, np.arange(N * (N + 2)) + 1 - n * n - n  # n, m of the flat entries


def _snm(N):
    """s_nm = sqrt(n(n+1)(2n+1)(n-m)!/(n+m)!) of one block."""
    n, m = _degrees(N)
    lg = np.array([math.lgamma(i + 1.0) for i in range(2 * N + 1)])
    return np.exp(0.5 * (np.log(n * (n + 1.0) * (2 * n + 1.0)) + lg[n - m] - lg[n + m]))


def _order(case):
    """The layout's order N: that of the largest radius of the law, so that one layout serves all its clusters."""
    return int(lmax_rule(np.array([1.0 if case["gen"] == "uniform" else 3.0]), case["wavelength"])[0])


def _vectors(cls, seed, nrhs, N):
    """Normalised coefficient vectors [nrhs, spheres, 2, N(N+2)]: order one up to the size parameter."""
    lmax = np.concatenate([c["lmax"] for c in cls])
    size = np.concatenate([c["k"] * c["radii"] for c in cls])
    n, _ = _degrees(N)
    env = (n[None, :] <= lmax[:, None]) / (1.0 + (n[None, :] / (size[:, None] + 1.0)) ** 8)
    rng = np.random.default_rng(seed + 77)
    v = rng.standard_normal((nrhs, len(lmax), 2, N * (N + 2), 2)).view(np.complex128)[..., 0]
    return v * env[None, :, None, :]


_work_stream = []


def _stream():
    """The program's one work stream."""
    if not _work_stream:
        _work_stream.append(torch.cuda.Stream())
    return _work_stream[0]


def prepare(case, seed):
    cls = _clusters(case, seed)
    c = cls[0]
    kind = case["kind"]
    nrhs = case.get("nrhs", 1)
    N = _order(case)
    if kind == "multi":
        s = ClusterBatch(cls, c["k"], n_global=N)
    else:
        s = MultiSphereSolver(c["centres"], c["radii"], c["m_rel"], c["k"], n_global=N, lmax=c["lmax"],
                              use_fmm=case.get("fmm", False), leaf_size=case.get("leaf", 32),
                              workspace_mb=16384, precision="mixed" if case.get("mixed") else "fp64")
    xh = _vectors(cls, seed, nrhs, N)
    snm = _snm(N)
    st = dict(case=case, solver=s, snm=snm, shape=(-1, 2, N * (N + 2)))
    if kind == "solve":
        rng = np.random.default_rng(seed)
        alpha, beta = rng.uniform(0.0, math.pi), rng.uniform(0.0, 2.0 * math.pi)
        st["rhs"] = s.get_vector_b_dir(alpha, beta)
        st["p"] = s.plane_wave(alpha, beta)
    elif kind == "far":
        st["x"] = (xh / snm).reshape(-1)
        st["theta"], st["phi"] = _grid(case)
    elif kind == "host":
        st["x"] = (xh / snm).reshape(-1)
    else:
        st["stream"] = _stream()
        with torch.cuda.stream(st["stream"]):
            st["x"] = torch.from_numpy((xh / snm).reshape(nrhs, -1)).to("cuda")
            st["b"] = torch.empty_like(st["x"])
            st["snm"] = torch.from_numpy(snm).to("cuda")
        s.set_stream(st["stream"].cuda_stream)
    return st


def _grid(case):
    th = np.linspace(0.0, math.pi, case["ntheta"])
    ph = np.arange(case["nphi"]) * (2.0 * math.pi / case["nphi"])
    return np.repeat(th, case["nphi"]), np.tile(ph, case["ntheta"])


def run(st):
    case, s = st["case"], st["solver"]
    kind = case["kind"]
    if kind == "host":
        return s.calculate_vector_b(st["x"]).reshape(st["shape"]) * st["snm"]
    if kind == "solve":
        x, _ = s.solve(st["rhs"], restart=case["restart"], tol=case["tol"])
        return x.reshape(st["shape"]) * st["snm"], np.array(s.cross_sections(x, st["p"]))
    if kind == "far":
        return s.far_field(st["x"], st["theta"], st["phi"])
    x, b = st["x"], st["b"]
    with torch.cuda.stream(st["stream"]):
        if case.get("nrhs", 1) > 1:
            s.calculate_vector_b_batch_device(x.data_ptr(), b.data_ptr(), case["nrhs"])
        elif case.get("graph"):
            s.calculate_vector_b_graph_device(x.data_ptr(), b.data_ptr())
        else:
            s.calculate_vector_b_device(x.data_ptr(), b.data_ptr())
        out = b.view(st["shape"]) * st["snm"]
        return out.to(torch.complex64) if case.get("mixed") else out


def work(case):
    """Vectors in and out; the flops of one rotate - shift - rotate back translation (64/3 L^3) per
    sphere pair that is applied directly, per sphere 27 leaf boxes' worth of them under the MLFMM."""
    k = 2.0 * math.pi / case["wavelength"]
    r = 0.65 if case["gen"] == "uniform" else 1.15
    x, xmax = k * r, k * (1.0 if case["gen"] == "uniform" else 3.0)
    L, N = x + 4.0 * x ** (1.0 / 3.0) + 2.0, xmax + 4.0 * xmax ** (1.0 / 3.0) + 2.0
    ns, pairs = case.get("n", 0), 0
    if case["kind"] == "multi":
        mean = 0.5 * (case["n_lo"] + case["n_hi"])
        ns, pairs = case["clusters"] * mean, case["clusters"] * mean * (mean - 1)
    elif case["kind"] == "far":
        ndir = case["ntheta"] * case["nphi"]
        return dict(bytes=32.0 * ns * N * N + 48.0 * ndir, flops=32.0 * ns * L * L * ndir)
    elif case.get("fmm"):
        pairs = ns * min(ns - 1, 27.0 * case["leaf"] / 2.0)
    else:
        pairs = ns * (ns - 1)
    nrhs = case.get("nrhs", 1)
    products = 10 if case["kind"] == "solve" else 1
    return dict(bytes=64.0 * ns * N * (N + 2) * nrhs, flops=64.0 / 3.0 * L ** 3 * pairs * nrhs * products)


# -- 64-bit reference -----------------------------------------------------------
def _bessel(x, nmax):
    """j_n(x), y_n(x), n = 0..nmax, for an array x: Miller's recurrence downward, y upward."""
    x = np.asarray(x, dtype=np.float64)
    j, y = np.zeros((nmax + 1,) + x.shape), np.zeros((nmax + 1,) + x.shape)
    top = int(max(nmax, x.max())) + 40 + int(math.sqrt(50.0 * max(nmax, x.max())))
    fp, f = np.zeros_like(x), np.full_like(x, 1e-280)
    for n in range(top, 0, -1):
        fp, f = f, (2 * n + 1) / x * f - fp
        if n - 1 <= nmax:
            j[n - 1] = f
        big = np.abs(f) > 1e200
        if big.any():
            sc = np.where(big, 1e-200, 1.0)
            f, fp = f * sc, fp * sc
            j *= sc
    j0, j1 = np.sin(x) / x, np.sin(x) / x ** 2 - np.cos(x) / x
    j *= np.where(np.abs(j0) > np.abs(j1), j0 / j[0], j1 / j[min(1, nmax)])
    y[0] = -np.cos(x) / x
    if nmax:
        y[1] = -np.cos(x) / x ** 2 - np.sin(x) / x
    for n in range(1, nmax):
        y[n + 1] = (2 * n + 1) / x * y[n] - y[n - 1]
    return j, y


def _mie(x, m, N):
    """Lorenz-Mie a_n, b_n (n = 1..N) of each sphere, logarithmic derivatives downward."""
    z = m * x
    top = int(max(N, np.abs(z).max())) + 30
    D, d = np.zeros((N + 1,) + x.shape, complex), np.zeros_like(z)
    for n in range(top, 0, -1):
        d = n / z - 1.0 / (d + n / z)
        if 1 <= n - 1 <= N:
            D[n - 1] = d
    j, y = _bessel(x, N)
    h = j + 1j * y
    n = np.arange(1, N + 1)[:, None]
    out = []
    for f in (D[1:] / m, D[1:] * m):
        t = f + n / x
        out.append((t * j[1:] - j[:-1]) / (t * h[1:] - h[:-1]))
    return out


def _legendre(N, mu, orthonormal=True):
    """P[m][n] at mu, n >= m, orthonormal on [-1, 1] and without the Condon-Shortley phase; without
    ``orthonormal`` the m = 0 row only, as Legendre polynomials."""
    if not orthonormal:
        P = np.ones((N + 1,) + mu.shape)
        for n in range(1, N + 1):
            P[n] = mu if n == 1 else ((2 * n - 1) * mu * P[n - 1] - (n - 1) * P[n - 2]) / n
        return P
    P = np.zeros((N + 1, N + 1) + mu.shape)
    s, d = np.sqrt(1.0 - mu * mu), np.full_like(mu, math.sqrt(0.5))
    for m in range(N + 1):
        if m:
            d = d * s * math.sqrt((2 * m + 1.0) / (2 * m))
        P[m, m] = d
        for n in range(m + 1, N + 1):
            a = math.sqrt((4.0 * n * n - 1) / (n * n - m * m))
            b = math.sqrt(((n - 1.0) ** 2 - m * m) / (4.0 * (n - 1) ** 2 - 1)) if n > m + 1 else 0.0
            P[m, n] = a * (mu * P[m, n - 1] - (b * P[m, n - 2] if n > m + 1 else 0.0))
    return P


def _direct_exact(cls, xh, N):
    """x + T A x in the normalised basis over all pairs of each cluster: scalar coaxial integrals
    over products of three Legendre functions (each Hankel order on its own, selection rules
    exact), the vector relation, and rotations from the eigenvectors of J_y."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    k = cls[0]["k"]
    T = lambda a: torch.as_tensor(a, device=dev)  # noqa: E731
    first = np.cumsum([0] + [len(c["radii"]) for c in cls])
    pos = np.concatenate([c["centres"] for c in cls])
    lmax = np.concatenate([c["lmax"] for c in cls])
    tgt = np.concatenate([np.repeat(np.arange(a, b), b - a) for a, b in zip(first, first[1:])])
    src = np.concatenate([np.tile(np.arange(a, b), b - a) for a, b in zip(first, first[1:])])
    tgt, src = tgt[tgt != src], src[tgt != src]
    mu, w = np.polynomial.legendre.leggauss(2 * N + 4)
    V, Pp = T(_legendre(N + 1, mu)), T(_legendre(2 * N + 1, mu, False) * w)
    n_, v_, p_ = np.ogrid[:N + 2, :N + 1, :2 * N + 2]
    sel = T(((p_ >= abs(n_ - v_)) & (p_ <= n_ + v_) & ((n_ + v_ + p_) % 2 == 0)).astype(float))
    G = [torch.einsum("nq,vq,pq->nvp", V[m], V[m, :N + 1], Pp) * sel for m in range(N + 1)]
    rot = []
    for n in range(N + 1):
        q = np.arange(-n, n)
        up = np.sqrt(n * (n + 1.0) - q * (q + 1))
        J = np.diag(-0.5j * up, -1) + np.diag(0.5j * up, 1)  # J_y
        rot.append(T(np.linalg.eigh(J)[1]))
    X = T(xh)
    X = torch.stack([X[:, :, 0] + X[:, :, 1], X[:, :, 0] - X[:, :, 1]], dim=2)  # x_+, x_-
    acc = torch.zeros_like(X)
    nn = torch.arange(1, N + 1, device=dev, dtype=torch.float64)
    step = max(1, int(2e8 // ((N + 2) ** 2 * 64 + 16 * (N + 1) ** 3)))
    for c0 in range(0, len(tgt), step):
        jt, js = tgt[c0:c0 + step], src[c0:c0 + step]
        d = pos[jt] - pos[js]
        r = np.sqrt((d * d).sum(1))
        th, ph = T(np.arctan2(np.hypot(d[:, 0], d[:, 1]), d[:, 2])), T(np.arctan2(d[:, 1], d[:, 0]))
        t = T(k * r)
        jn, yn = _bessel(k * r, 2 * N + 1)
        pp = np.arange(2 * N + 2)
        H = T((jn + 1j * yn) * ((1j ** pp) * (2 * pp + 1))[:, None])
        B, R = len(jt), X.shape[0]
        Y = torch.zeros((B, R, 2, N + 1, 2 * N + 1), dtype=torch.complex128, device=dev)
        dm = [None]
        Xs = X[:, T(js)].transpose(0, 1)
        for n in range(1, N + 1):
            m = torch.arange(-n, n + 1, device=dev)
            ev = torch.exp(-1j * th[:, None] * m)
            D = torch.matmul(rot[n][None] * ev[:, None, :], rot[n].conj().T.contiguous()).real.to(torch.complex128)
            dm.append(D)
            ein = torch.exp(1j * ph[:, None] * m)
            xs = Xs[..., n * n - 1:n * n + 2 * n] * ein[:, None, None, :]
            Y[:, :, :, n, N - n:N + n + 1] = torch.matmul(xs.reshape(B, 2 * R, -1), D.transpose(1, 2).contiguous()
                                                          ).reshape(B, R, 2, -1)
        Z = torch.zeros_like(Y)
        for m in range(N + 1):
            q = max(m, 1)
            g = G[m].reshape(-1, 2 * N + 2)
            I = torch.complex(g @ H.real, g @ H.imag).reshape(N + 2, N + 1, B).permute(2, 0, 1).contiguous()
            f0 = torch.sqrt(nn * (nn + 1))
            am = lambda x: torch.sqrt(((x + 1) ** 2 - m * m).clamp(min=0) / ((2 * x + 1) * (2 * x + 3)))  # noqa: E731
            fp = t[:, None] * am(nn) * torch.sqrt(nn / (nn + 1))
            fm = t[:, None] * am(nn - 1) * torch.sqrt((nn + 1) / nn)
            fb = t[:, None] * m / f0
            for s in ([1, -1] if m else [1]):
                y = Y[:, :, :, 1:, N + s * m] / f0
                y[..., :q - 1] = 0.0
                u = torch.matmul(I[:, :, 1:], y.reshape(B, 2 * R, N).transpose(1, 2).contiguous()).transpose(1, 2)
                u = u.reshape(B, R, 2, N + 2)
                e = [x[:, None, None, :] for x in (fp, fm, fb)]
                um = u[..., :N] if m == 0 else torch.cat([torch.zeros_like(u[..., :m]), u[..., m:N]], -1)
                A = f0 * u[..., 1:N + 1] + 1j * e[0] * u[..., 2:] - 1j * e[1] * um
                Bc = 1j * e[2] * u[..., 1:N + 1]
                sgn = torch.tensor([1.0, -1.0], device=dev)[:, None] * s
                z = A + sgn * Bc
                z[..., :q - 1] = 0.0
                Z[:, :, :, 1:, N + s * m] = z
        out = torch.zeros((B, R, 2, N * (N + 2)), dtype=torch.complex128, device=dev)
        for n in range(1, N + 1):
            m = torch.arange(-n, n + 1, device=dev)
            z = Z[:, :, :, n, N - n:N + n + 1].reshape(B, 2 * R, -1)
            out[..., n * n - 1:n * n + 2 * n] = (torch.matmul(z, dm[n]).reshape(B, R, 2, -1)
                                                 * torch.exp(-1j * ph[:, None] * m)[:, None, None, :])
        acc.index_add_(1, T(jt), out.transpose(0, 1).contiguous())
    acc = 0.5 * torch.stack([acc[:, :, 0] + acc[:, :, 1], acc[:, :, 0] - acc[:, :, 1]], dim=2)
    size = np.concatenate([c["k"] * c["radii"] for c in cls])
    a, b = _mie(size, np.concatenate([c["m_rel"] for c in cls]), N)
    deg, _ = _degrees(N)
    mask = deg[None, :] <= lmax[:, None]
    ab = np.stack([a[deg - 1].T * mask, b[deg - 1].T * mask], axis=1)
    return (xh + (T(ab)[None] * acc).cpu().numpy()).reshape(-1, 2, N * (N + 2))


def _far_exact(case, c, xh, N):
    th, ph = _grid(case)
    deg, m = _degrees(N)
    am = np.abs(m)
    t1 = np.unique(th)
    P = _legendre(N + 1, np.cos(t1))
    sn = np.sin(t1)
    nn, mm = np.arange(N + 2)[None, :, None], np.arange(N + 2)[:, None, None]
    nrm = np.sqrt(2.0 / (2 * nn + 1.0))  # to sqrt((n-m)!/(n+m)!) P_n^m
    Q = P * nrm
    with np.errstate(divide="ignore", invalid="ignore"):
        pi = np.where(sn > 0, mm * Q / sn, 0.0)
    up, dn = np.zeros_like(Q), np.zeros_like(Q)
    up[:-1] = Q[1:]
    dn[1:] = Q[:-1]
    # d/dtheta of the normalised functions: half the difference of the neighbouring orders
    tau = 0.5 * (np.sqrt(np.clip((nn + mm) * (nn - mm + 1.0), 0, None)) * dn
                 - np.sqrt(np.clip((nn - mm) * (nn + mm + 1.0), 0, None)) * up)
    tau[0] = -np.sqrt(nn[0] * (nn[0] + 1.0)) * Q[1]
    pole = sn < 1e-9  # the poles: only |m| = 1, sqrt(n(n+1))/2 with alternating signs behind
    for i in np.nonzero(pole)[0]:
        pi[:, :, i] = tau[:, :, i] = 0.0
        h = 0.5 * np.sqrt(nn[0, :, 0] * (nn[0, :, 0] + 1.0))
        back = t1[i] > 1.0
        alt = (-1.0) ** nn[0, :, 0]
        pi[1, :, i] = -alt * h if back else h
        tau[1, :, i] = alt * h if back else h
    row = np.searchsorted(t1, th)
    sg = np.where((m < 0) & (am % 2 == 1), -1.0, 1.0)
    f = np.sqrt((2 * deg + 1.0) / (deg * (deg + 1.0)))
    tauv = (tau[am, deg] * (sg * f)[:, None]).T
    piv = (pi[am, deg] * (sg * f * np.where(m < 0, -1.0, 1.0))[:, None]).T
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    T = lambda a: torch.as_tensor(a, device=dev)  # noqa: E731
    X = T(xh[0])
    out = [[], []]
    for i in range(0, len(th), 2048):
        s = slice(i, i + 2048)
        rh = np.stack([np.sin(th[s]) * np.cos(ph[s]), np.sin(th[s]) * np.sin(ph[s]), np.cos(th[s])], 1)
        e = torch.exp(-1j * c["k"] * T(rh @ c["centres"].T))
        ab = torch.matmul(e, X.reshape(X.shape[0], -1)).reshape(-1, 2, N * (N + 2))
        em = torch.exp(1j * T(ph[s][:, None] * m[None, :]))
        ta, pa = T(tauv[row[s]]) * em, T(piv[row[s]]) * em
        out[0].append((1j * (ab[:, 0] * ta + ab[:, 1] * pa).sum(1)).cpu().numpy())
        out[1].append((-(ab[:, 0] * pa + ab[:, 1] * ta).sum(1)).cpu().numpy())
    return np.concatenate(out[0]), np.concatenate(out[1])


def exact(case, seed):
    """Direct products and far fields in 64 bits.  A solve ends at its tolerance and has no such
    value; an MLFMM product is compared with the sum over all pairs where that is short."""
    if case["kind"] == "solve" or (case.get("fmm") and case["n"] > (220 if case["gen"] == "lognormal" else 400)):
        return None
    cls = _clusters(case, seed)
    N = _order(case)
    xh = _vectors(cls, seed, case.get("nrhs", 1), N)
    if case["kind"] == "far":
        return _far_exact(case, cls[0], xh, N)
    return _direct_exact(cls, xh, N)
