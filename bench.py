"""Benchmark: MLFMM matvecs/s of the 2000-sphere cluster on one MI355X.

One step = one matvec b = (I + T A) x of the 2000-water-sphere cluster (lognormal
radii, median 1 um, sigma_g 1.5, clipped to [0.2, 3] um, volume fraction 1e-3,
lambda 550 nm, seed 2000) through the MLFMM (leaf <= 32 spheres, box truncation
L = kD + 1.8 d0^(2/3) (kD)^(1/3), d0 = 6), FP64, inputs resident in HBM.

``--config 3 [--wavelength 1.55]``: the same measurement on the 20000-sphere cluster
(radii uniform in [0.3, 1] um in a 100 um cube, 550 or 1550 nm) with GMRES(30).

Prints one JSON line (rank 0).  The CPU baseline times the oracle (the
reference's algorithm: full Gaunt/3j translation matrices per sphere pair,
regenerated every matvec) on a bounded sample of sphere pairs of the same
cluster and extrapolates to one direct matvec over all ordered pairs.
"""
import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

FP64_PEAK_TFLOPS = 78.6
FP32_PEAK_TFLOPS = 157.3
HBM_PEAK_TBS = 8.0
METRIC = "MLFMM matvecs/s & solves/s at rel. residual 1e-6; p50/p99 solve latency"


def snm_flat(N, ns):
    """s_nm = sqrt(n(n+1)(2n+1)(n-m)!/(n+m)!) over the flat vector (a and b blocks, ns spheres)."""
    from math import lgamma
    s = np.array([np.exp(0.5 * (np.log(n * (n + 1) * (2 * n + 1)) + lgamma(n - m + 1) - lgamma(n + m + 1)))
                  for n in range(1, N + 1) for m in range(-n, n + 1)])
    return np.tile(np.concatenate([s, s]), ns)


def roofline(kern, traffic, suffix):
    """The kernel group that takes longest against what bounds it: the matrix cores (FP64; FP32 for
    the groups named so) or, where its HBM bytes are known and take longer at their peak, HBM.
    kern: {name: (total ms, launches, algorithmic flops)}; traffic: bytes per launch by name and suffix."""
    dom = max(kern, key=lambda k: kern[k][0])
    tot_ms, launches, fl = kern[dom]
    t = traffic.get(dom + suffix)
    per_launch = t["read"] + t["write"] if t else None
    peak = FP32_PEAK_TFLOPS if dom.endswith("_f32") else FP64_PEAK_TFLOPS
    tflops = fl / (tot_ms * 1e-3) / 1e12
    tbs = per_launch * launches / (tot_ms * 1e-3) / 1e12 if t else 0.0
    hbm = tbs / HBM_PEAK_TBS > tflops / peak
    got, top = (tbs, HBM_PEAK_TBS) if hbm else (tflops, peak)
    return {"bound": "hbm" if hbm else "mfma", "kernel": dom, "achieved": round(got, 3), "peak": top,
            "unit": "TB/s" if hbm else "TFLOP/s", "frac": round(got / top, 4), "tflops": round(tflops, 3),
            "traffic": per_launch, "traffic_unit": "bytes/launch", "launches": launches,
            "avg_launch_ms": round(tot_ms / launches, 4), "algorithmic_flops_per_launch": fl / launches}


def cpu_model():
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return None


def cpu_baseline(cluster, npairs, threads, affinity):
    from oracle import oracle as O
    ns = len(cluster["radii"])
    N = int(cluster["lmax"].max())
    rng = np.random.default_rng(12345)
    tgt = rng.integers(0, ns, npairs).astype(np.int32)
    src = ((tgt + 1 + rng.integers(0, ns - 1, npairs)) % ns).astype(np.int32)
    an = np.full((ns, N), 0.5 + 0.1j)
    bn = an.copy()
    x = np.ones(ns * 2 * N * (N + 2), dtype=np.complex128)
    t0 = time.perf_counter()
    O.matvec_pairs(cluster["centres"], cluster["lmax"], N, an, bn, cluster["k"], x, tgt, src, nthreads=threads)
    dt = time.perf_counter() - t0
    pairs_per_s = npairs / dt
    return {"value": pairs_per_s / (ns * (ns - 1)), "unit": "matvecs/s", "cores": threads, "kind": "port",
            "cpu_model": cpu_model(), "nproc": os.cpu_count(), "affinity_cpus": affinity,
            "omp_proc_bind": os.environ.get("OMP_PROC_BIND"),
            "sample": f"{npairs} random ordered sphere pairs of the same {ns}-sphere cluster through the oracle "
                      f"(full Xu A/B by the Gaunt/3j formula per pair, dense apply) in {dt:.1f} s on {threads} "
                      f"threads, extrapolated to one direct matvec over all {ns * (ns - 1)} ordered pairs"}


def solution_errors(s, x64, x32):
    """Mixed-precision solution against the FP64 one: coefficients (normalised basis),
    C_sca/C_ext/C_abs of the +z x-polarised plane wave, far field on the 181 x 36
    (theta, phi) grid (lib_mie_ss_helper_functions.f90:1380-1475)."""
    import math
    S = snm_flat(s.n_global, s.n_spheres)
    p = s.plane_wave(0.0, 0.0)
    cs64 = np.array(s.cross_sections(x64, p))
    cs32 = np.array(s.cross_sections(x32, p))
    th = np.repeat(np.linspace(0.0, math.pi, 181), 36)
    ph = np.tile(np.linspace(0.0, 2 * math.pi, 36, endpoint=False), 181)
    f64 = np.concatenate(s.far_field(x64, th, ph))
    f32 = np.concatenate(s.far_field(x32, th, ph))
    return {"coefficients": float(np.linalg.norm((x32 - x64) * S) / np.linalg.norm(x64 * S)),
            "c_sca_ext_abs": [float(v) for v in np.abs(cs32 - cs64) / np.abs(cs64)],
            "far_field_181x36": float(np.max(np.abs(f32 - f64)) / np.max(np.abs(f64))),
            "c_sca_ext_abs_fp64_um2": [float(v) for v in cs64]}


def solve_latency(seeds, x0, max_iter, log, n=None, precision="fp64"):
    """End-to-end request latency on fresh contexts: create (octree, Mie, plan) + first
    matvec's table generation + GMRES(50) to 1e-6 from the single-sphere solution
    (precision 'mixed': FP32 box products in the Arnoldi steps, FP64 true residuals)."""
    import torch
    from itofoggysim_amd import MultiSphereSolver, config_cluster
    runs = []
    for seed in seeds:
        c = config_cluster(2, replica=seed - 2000, n=n)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        s = MultiSphereSolver(c["centres"], c["radii"], c["m_rel"], c["k"], lmax=c["lmax"], use_fmm=True,
                              leaf_size=32, fmm_d0=6.0)
        t_build = time.perf_counter() - t0
        rhs = torch.from_numpy(s.get_vector_b()).to("cuda")
        xs = rhs.clone() if x0 == "single" else torch.zeros_like(rhs)
        torch.cuda.synchronize()
        info = s.solve_device(rhs.data_ptr(), xs.data_ptr(), restart=50, max_iter=max_iter, tol=1e-6,
                              use_x0=x0 == "single", verbose=False, precision=precision)
        total = time.perf_counter() - t0
        s.close()
        del rhs, xs
        runs.append({"seed": seed, "create_s": round(t_build, 3), "solve_s": round(info["seconds"], 3),
                     "total_s": round(total, 3), "iterations": info["iterations"], "converged": info["converged"],
                     "rel_residual": info["rel_residual"], "rel_residual_flat": info["rel_residual_flat"]})
        print(f"# latency {precision} seed {seed}: {total:.1f} s end to end ({info['iterations']} matvecs, "
              f"residual {info['rel_residual']:.2e})", file=log, flush=True)
    tot = sorted(r["total_s"] for r in runs)
    # p50 / p99 by linear interpolation over the samples
    return {"samples": len(runs), "p50_s": round(float(np.percentile(tot, 50)), 3),
            "p99_s": round(float(np.percentile(tot, 99)), 3),
            "solves_per_s": round(len(runs) / sum(tot), 5) if all(r["converged"] for r in runs) else None,
            "runs": runs}


def fibonacci_directions(n):
    """n propagation directions (alpha, beta) on a Fibonacci sphere."""
    i = np.arange(n) + 0.5
    return np.arccos(1.0 - 2.0 * i / n), np.mod(i * np.pi * (3.0 - np.sqrt(5.0)), 2.0 * np.pi)


def config4(args):
    """Batched right-hand sides and many clusters per launch:
    (a) a 5000-sphere cluster (radii U[0.3,1] um, 20-sphere number density, 550 nm, MLFMM
        leaf <= 32, d0 = 6): matvec time per right-hand side for 1, 8 and 32 columns in
        one batched product (FP64 and mixed), and the first --c4-dirs of 128 Fibonacci
        directions x TM/TE solved in lock step (mixed, GMRES(30) to 1e-6);
    (b) --c4-clusters independent clusters (N uniform in [10, 200], the same generator)
        in one context: one matvec launch for all (eager and HIP-graph replay), and all
        solved by per-cluster GMRES(30) to 1e-6 in lock step (graph-captured products)."""
    import torch
    from itofoggysim_amd import ClusterBatch, MultiSphereSolver, make_cluster
    out = {"metric": METRIC, "n_gpus": 1, "higher_is_better": True, "dtype": "f64", "data": "synthetic",
           "config": {"workload": "config 4: batched right-hand sides (5000 spheres) and many clusters per launch"}}
    c = make_cluster(5000, ("uniform", 0.3, 1.0), side=10.0 * (5000 / 20.0) ** (1.0 / 3.0), seed=4000)
    t0 = time.perf_counter()
    s = MultiSphereSolver(c["centres"], c["radii"], c["m_rel"], c["k"], lmax=c["lmax"], use_fmm=True, leaf_size=32,
                          fmm_d0=6.0)
    out["cluster5000"] = {"create_s": round(time.perf_counter() - t0, 3), "unknowns_flat": s.n,
                          "lmax_range": [int(c["lmax"].min()), int(c["lmax"].max())]}
    print(f"# 5000 spheres: {s.n} unknowns, created in {out['cluster5000']['create_s']} s", file=sys.stderr,
          flush=True)
    gen = torch.Generator(device="cpu").manual_seed(5)
    st = torch.cuda.Stream()
    s.set_stream(st.cuda_stream)
    per_rhs = {}
    for prec in ("fp64", "mixed"):
        s.set_precision(prec)
        for nr in (1, 8, 32):
            X = torch.randn(nr, s.n, dtype=torch.complex128, generator=gen).to("cuda")
            B = torch.empty_like(X)
            torch.cuda.synchronize()
            s.calculate_vector_b_batch_device(X.data_ptr(), B.data_ptr(), nr)  # tables, buffers
            st.synchronize()
            t0 = time.perf_counter()
            s.calculate_vector_b_batch_device(X.data_ptr(), B.data_ptr(), nr)
            st.synchronize()
            dt = time.perf_counter() - t0
            per_rhs[f"{prec}_nrhs{nr}_ms_per_rhs"] = round(1000 * dt / nr, 2)
            print(f"# 5000 spheres {prec}: {nr} columns {1000 * dt:.0f} ms ({1000 * dt / nr:.1f} ms per rhs)",
                  file=sys.stderr, flush=True)
            del X, B
    s.set_precision("fp64")
    s.set_stream(0)
    out["cluster5000"]["matvec"] = per_rhs
    al, be = fibonacci_directions(128)
    nd = args.c4_dirs
    rhs = np.stack([s.get_vector_b_dir(al[i], be[i], te=te) for i in range(nd) for te in (False, True)])
    t0 = time.perf_counter()
    X, infos = s.solve_batch(rhs, restart=30, tol=1e-6, max_iter=400, precision="mixed", raise_on_noconv=False,
                             verbose=True)
    dt = time.perf_counter() - t0
    out["cluster5000"]["block_solve"] = {
        "rhs": 2 * nd, "of": 256, "precision": "mixed", "seconds": round(dt, 3),
        "solves_per_s": round(2 * nd / dt, 4), "all_converged": all(i["converged"] for i in infos),
        "iterations": [i["iterations"] for i in infos], "max_rel_residual": max(i["rel_residual"] for i in infos),
        "extrapolated_256_rhs_s": round(dt * 256 / (2 * nd), 1)}
    print(f"# 5000 spheres: {2 * nd} right-hand sides solved in lock step in {dt:.1f} s", file=sys.stderr,
          flush=True)
    # the same right-hand sides by block GMRES (one Krylov space of 30 block steps x 2 nd vectors)
    t0 = time.perf_counter()
    Xb, ib = s.solve_block(rhs, restart=30, tol=1e-6, max_iter=400, precision="mixed", raise_on_noconv=False,
                           verbose=True)
    dtb = time.perf_counter() - t0
    S = snm_flat(s.n_global, s.n_spheres)
    out["cluster5000"]["block_gmres"] = {
        "rhs": 2 * nd, "precision": "mixed", "seconds": round(dtb, 3), "solves_per_s": round(2 * nd / dtb, 4),
        "products_per_rhs": ib[0]["iterations"], "all_converged": all(i["converged"] for i in ib),
        "max_rel_residual": max(i["rel_residual"] for i in ib),
        "max_diff_vs_lock_step": float(max(np.linalg.norm((Xb[r] - X[r]) * S) / np.linalg.norm(X[r] * S)
                                           for r in range(2 * nd)))}
    print(f"# 5000 spheres: {2 * nd} right-hand sides by block GMRES in {dtb:.1f} s", file=sys.stderr, flush=True)
    s.close()
    # (b) many clusters in one context
    rng = np.random.default_rng(256)
    sizes = rng.integers(10, 201, args.c4_clusters)
    t0 = time.perf_counter()
    cls = [make_cluster(int(n), ("uniform", 0.3, 1.0), side=10.0 * (n / 20.0) ** (1.0 / 3.0), seed=5000 + i)
           for i, n in enumerate(sizes)]
    t_gen = time.perf_counter() - t0
    t0 = time.perf_counter()
    mb = ClusterBatch(cls, cls[0]["k"])
    t_create = time.perf_counter() - t0
    print(f"# {len(cls)} clusters ({mb.n_spheres} spheres, {mb.n} unknowns): generated in {t_gen:.1f} s, "
          f"context in {t_create:.1f} s", file=sys.stderr, flush=True)
    x = torch.randn(mb.n, dtype=torch.complex128, generator=gen).to("cuda")
    b = torch.empty_like(x)
    torch.cuda.synchronize()
    mb.set_stream(st.cuda_stream)
    times = {}
    for mode in ("eager", "graph"):
        f = mb.calculate_vector_b_device if mode == "eager" else mb.calculate_vector_b_graph_device
        for _ in range(2):
            f(x.data_ptr(), b.data_ptr())
        st.synchronize()
        t0 = time.perf_counter()
        for _ in range(3):
            f(x.data_ptr(), b.data_ptr())
        st.synchronize()
        times[mode] = (time.perf_counter() - t0) / 3
    mb.set_stream(0)
    rhs = mb.get_vector_b()
    t0 = time.perf_counter()
    xs, infos = mb.solve(rhs, restart=30, tol=1e-6, max_iter=400, x0=rhs, graph=True, raise_on_noconv=False,
                         verbose=True)
    dt = time.perf_counter() - t0
    out["clusters"] = {
        "clusters": len(cls), "spheres": mb.n_spheres, "unknowns_flat": mb.n, "n_range": [int(sizes.min()),
                                                                                           int(sizes.max())],
        "generate_s": round(t_gen, 2), "create_s": round(t_create, 2),
        "matvec_ms": {k: round(1000 * v, 2) for k, v in times.items()},
        "solve_s": round(dt, 3), "solves_per_s": round(len(cls) / dt, 3),
        "all_converged": all(i["converged"] for i in infos),
        "iterations_max": max(i["iterations"] for i in infos),
        "max_rel_residual": max(i["rel_residual"] for i in infos)}
    out["value"] = out["clusters"]["solves_per_s"]
    out["unit"] = "solves/s"
    print(f"# {len(cls)} clusters solved in {dt:.1f} s", file=sys.stderr, flush=True)
    mb.close()
    return out


def main():
    # the CPU baseline's OpenMP threads: all cores, bound close (read at libgomp load; the
    # binding pins the main thread, so the CPU set is read first)
    affinity = len(os.sched_getaffinity(0))
    os.environ.setdefault("OMP_PROC_BIND", "close")
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--cpu-pairs", type=int, default=400)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-solve", action="store_true", help="skip the GMRES(50) solve to 1e-6")
    ap.add_argument("--solve-max-iter", type=int, default=None, help="default 100 (config 2), 400 (config 3)")
    ap.add_argument("--x0", choices=("single", "zero"), default="single",
                    help="GMRES initial guess: the single-sphere solution T_j p_j, i.e. the right-hand side "
                         "(lib_mie_multi_sphere.f90:134-138), or zero")
    ap.add_argument("--n", type=int, default=2000, help="sphere count (default: the 2000-sphere cluster)")
    ap.add_argument("--config", type=int, choices=(2, 3, 4), default=2,
                    help="2: the 2000-sphere lognormal cluster (default); 3: 20000 spheres U[0.3,1] um at the "
                         "20-sphere cluster's number density (100 um cube), GMRES(30); 4: batched right-hand "
                         "sides of a 5000-sphere cluster and 256 clusters of N in [10, 200] in one context")
    ap.add_argument("--c4-dirs", type=int, default=4,
                    help="config 4: incidence directions (x TM/TE) solved in lock step out of the 128")
    ap.add_argument("--c4-clusters", type=int, default=256, help="config 4: independent clusters in one context")
    ap.add_argument("--wavelength", type=float, default=0.55, help="config 3 only: 0.55 or 1.55 um")
    ap.add_argument("--serve-requests", type=int, default=16,
                    help="serving workload: Poisson arrivals of this many requests (0 skips it)")
    ap.add_argument("--serve-rate", type=float, default=2.0, help="serving arrival rate, requests/s")
    ap.add_argument("--serve-nmax", type=int, default=500,
                    help="largest cluster of the serving workload (the stated workload goes to 20000)")
    ap.add_argument("--serve-dirs", type=int, default=8, help="most incidence directions of a serving request")
    ap.add_argument("--serve-slots", type=int, default=4,
                    help="serving worker slots (requests running at once; 4 = the process's hardware queues)")
    ap.add_argument("--serve-verbose", action="store_true",
                    help="serving progress on stderr (each request's GMRES steps and completion)")
    ap.add_argument("--latency-seeds", type=int, default=2,
                    help="clusters (seeds 2000, 2001, ...) for the end-to-end solve latency; 0 skips it")
    ap.add_argument("--copy-probe", action="store_true",
                    help="only run a plain 1 GiB device copy (calibrates FETCH_SIZE / WRITE_SIZE counters)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: this build measures one GPU only (asked for {args.gpus}); run with --gpus 1",
              file=sys.stderr)
        sys.exit(2)

    import torch
    if args.copy_probe:
        nbytes = 1 << 30
        src = torch.ones(nbytes // 8, dtype=torch.float64, device="cuda")
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        print(json.dumps({"copy_probe_bytes_read": nbytes, "copy_probe_bytes_written": nbytes, "dispatches": 3}))
        return
    from itofoggysim_amd import MultiSphereSolver, config_cluster

    if args.config == 4:
        print(json.dumps(config4(args)))
        return
    if args.config == 3:
        c = config_cluster(3, wavelength=args.wavelength)
        args.latency_seeds = 0
        args.serve_requests = 0
        restart = 30
        args.solve_max_iter = args.solve_max_iter or 400
        workload = (f"MLFMM matvec of the 20000-sphere water cluster (r uniform in [0.3,1] um, 100 um cube, "
                    f"lambda {args.wavelength * 1000:.0f} nm, m = {c['m_rel'][0]:.6g}), leaf <= 32, box L = kD + "
                    f"1.8 d0^(2/3) (kD)^(1/3) with d0 = 6, FP64")
    else:
        c = config_cluster(2, n=args.n if args.n != 2000 else None)
        restart = 50
        args.solve_max_iter = args.solve_max_iter or 100
        workload = ("MLFMM matvec of the 2000-sphere water cluster (lognormal r, median 1 um, sigma_g 1.5, "
                    "[0.2,3] um, volume fraction 1e-3, lambda 550 nm), leaf <= 32, box L = kD + 1.8 d0^(2/3)"
                    " (kD)^(1/3) with d0 = 6, FP64")
    t0 = time.perf_counter()
    s = MultiSphereSolver(c["centres"], c["radii"], c["m_rel"], c["k"], lmax=c["lmax"], use_fmm=True,
                          leaf_size=32, fmm_d0=6.0)
    build_s = time.perf_counter() - t0
    counts, levels = s.fmm_stats()
    flops_mv, bytes_mv = s.matvec_cost()
    print(f"# built: {s.n_spheres} spheres, N={s.n_global}, vector {s.n}, levels L={levels}, {counts}, "
          f"{build_s:.2f} s", file=sys.stderr, flush=True)

    st = torch.cuda.Stream()
    gen = torch.Generator(device="cpu").manual_seed(2000)
    x = torch.randn(s.n, dtype=torch.complex128, generator=gen).to("cuda")
    b = torch.empty_like(x)
    with torch.cuda.stream(st):
        s.set_stream(st.cuda_stream)
        for i in range(args.warmup):
            s.calculate_vector_b_device(x.data_ptr(), b.data_ptr())
            st.synchronize()
            print(f"# warmup {i + 1}/{args.warmup} done", file=sys.stderr, flush=True)
        torch.cuda.synchronize()
        e0 = torch.cuda.Event(enable_timing=True)
        e1 = torch.cuda.Event(enable_timing=True)
        w0 = time.perf_counter()
        e0.record(st)
        for i in range(args.steps):
            s.calculate_vector_b_device(x.data_ptr(), b.data_ptr())
        e1.record(st)
        st.synchronize()
        torch.cuda.synchronize()
        wall = time.perf_counter() - w0
        ms = e0.elapsed_time(e1) / args.steps
        print(f"# timed {args.steps} steps: {ms:.1f} ms/step (wall {wall:.2f} s)", file=sys.stderr, flush=True)
        # per-kernel profile of one extra matvec (HIP events on the launch stream)
        s.profile(True)
        s.calculate_vector_b_device(x.data_ptr(), b.data_ptr())
        prof = s.profile_read()
        s.profile(False)
        # the same matvec with FP32 matrix-core box translations (ifs_set_precision)
        s.set_precision("mixed")
        b32 = torch.empty_like(x)
        s.calculate_vector_b_device(x.data_ptr(), b32.data_ptr())
        st.synchronize()
        e0.record(st)
        for i in range(args.steps):
            s.calculate_vector_b_device(x.data_ptr(), b32.data_ptr())
        e1.record(st)
        st.synchronize()
        ms32 = e0.elapsed_time(e1) / args.steps
        s.profile(True)
        s.calculate_vector_b_device(x.data_ptr(), b32.data_ptr())
        prof32 = s.profile_read()
        s.profile(False)
        # accuracy of the mixed matvec on an input random in the normalised basis (x = x_hat / s_nm;
        # the timed x is random in the flat basis, whose normalised entries span 1e+-80)
        snm = torch.from_numpy(snm_flat(s.n_global, s.n_spheres)).to("cuda")
        xe = torch.randn(s.n, dtype=torch.complex128, generator=gen).to("cuda") / snm
        be32 = torch.empty_like(x)
        be64 = torch.empty_like(x)
        s.calculate_vector_b_device(xe.data_ptr(), be32.data_ptr())
        s.set_precision("fp64")
        s.calculate_vector_b_device(xe.data_ptr(), be64.data_ptr())
        st.synchronize()
        print(f"# mixed: {ms32:.1f} ms/step", file=sys.stderr, flush=True)
    finite = bool(torch.isfinite(b).all().item())
    # mixed vs FP64 matvec, relative in the normalised basis
    mixed_err = float(torch.linalg.norm((be32 - be64) * snm) / torch.linalg.norm((be64 - xe) * snm))

    # the scopes that report algorithmic flops; HBM bytes per launch of the largest kernels:
    # measured offline with FETCH_SIZE / WRITE_SIZE counter runs of this same workload, calibrated
    # on a plain copy (profiles/)
    kern = {k: v for k, v in prof.items() if v[2] > 0}
    traffic_file = "profiles/mlfmm_2000_spheres_traffic.json"
    traffic = {}
    if os.path.exists(os.path.join(ROOT, traffic_file)) and args.n == 2000 and args.config == 2:
        traffic = json.load(open(os.path.join(ROOT, traffic_file)))["bytes_per_dispatch"]
    roof = roofline(kern, traffic, "")
    roof["traffic_source"] = traffic_file if roof["traffic"] else None
    # the same launches counted in the per-translation unit of the reference's formulation
    # (unfolded rotations, coaxial operator [A B; B A] not decoupled): the coaxial shift
    # performs exactly half of that count, so its reference-unit rate is twice its own
    roof["achieved_reference_unit"] = round(2.0 * roof["tflops"], 3) if roof["kernel"] == "class_axial" else None
    roof["matvec_algorithmic_tflops"] = round(flops_mv / (ms * 1e-3) / 1e12, 3)

    out = {
        "metric": METRIC,
        "value": round(1000.0 / ms, 6),
        "unit": "matvecs/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms, 3),
        "higher_is_better": True,
        "scaling": "strong",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic (seeded cluster generator, seed 2000; random seeded x)",
        "config": {
            "workload": workload,
            "n_spheres": s.n_spheres, "unknowns_flat": s.n, "box_L_per_level": levels, "translations": counts,
            "matvec_algorithmic_flop": flops_mv, "build_s": round(build_s, 3)},
        "roofline": roof,
        "kernels_ms": {k: round(v[0], 2) for k, v in prof.items()},
        "kernels_tflops": {k: round(v[2] / (v[0] * 1e-3) / 1e12, 2) for k, v in kern.items() if v[0] > 0},
        "finite": finite,
    }
    kern32 = {k: v for k, v in prof32.items() if v[2] > 0 and v[0] > 0}
    out["mixed"] = {
        "roofline": roofline(kern32, traffic, "_mixed"),
        "value": round(1000.0 / ms32, 6), "unit": "matvecs/s", "ms_per_step": round(ms32, 3),
        "speedup_vs_fp64": round(ms / ms32, 3),
        "rel_error_vs_fp64_normalised": mixed_err,
        "kernels_ms": {k: round(v[0], 2) for k, v in prof32.items()},
        "kernels_tflops": {k: round(v[2] / (v[0] * 1e-3) / 1e12, 2) for k, v in kern32.items()},
        "note": "M2M, L2L and M2L's class products as FP32 matrix-core products (FP32 accumulation) on the FP64 "
                "tables, plane-wave M2L tables in FP32; samples, sphere-level translations, T-apply and vectors "
                "FP64; FP32 peak 157.3 TFLOP/s"}
    if not args.no_solve:
        rhs = torch.from_numpy(s.get_vector_b()).to("cuda")
        # the single-sphere solution of (I + T A) x = T p is x_j = T_j p_j, the right-hand side itself
        xs = rhs.clone() if args.x0 == "single" else torch.zeros_like(rhs)
        torch.cuda.synchronize()
        with torch.cuda.stream(st):
            info = s.solve_device(rhs.data_ptr(), xs.data_ptr(), restart=restart, max_iter=args.solve_max_iter,
                                  tol=1e-6, use_x0=args.x0 == "single", verbose=True)
        torch.cuda.synchronize()
        x64 = xs.cpu().numpy()
        info["initial_guess"] = "single-sphere solution" if args.x0 == "single" else "zero"
        info["note"] = "tables generated in the warm-up matvec (steady-state solve)"
        out["solve"] = info
        out["solves_per_s_steady"] = 1.0 / info["seconds"] if info["converged"] else None
        xs = rhs.clone() if args.x0 == "single" else torch.zeros_like(rhs)
        torch.cuda.synchronize()
        with torch.cuda.stream(st):
            info32 = s.solve_device(rhs.data_ptr(), xs.data_ptr(), restart=restart, max_iter=args.solve_max_iter,
                                    tol=1e-6, use_x0=args.x0 == "single", verbose=True, precision="mixed")
        torch.cuda.synchronize()
        out["solve_mixed"] = info32
        out["solve_mixed"]["vs_fp64"] = solution_errors(s, x64, xs.cpu().numpy())
        out["solves_per_s_steady_mixed"] = 1.0 / info32["seconds"] if info32["converged"] else None
        del rhs, xs
    s.close()
    if not args.no_solve and args.latency_seeds > 0:
        torch.cuda.synchronize()
        seeds = [2000 + i for i in range(args.latency_seeds)]
        nn = args.n if args.n != 2000 else None
        lat = solve_latency(seeds, args.x0, args.solve_max_iter, sys.stderr, n=nn)
        out["solve_latency_s"] = {k: lat[k] for k in ("p50_s", "p99_s", "samples")}
        out["solves_per_s"] = lat["solves_per_s"]
        out["solve_latency_runs"] = lat["runs"]
        lat32 = solve_latency(seeds, args.x0, args.solve_max_iter, sys.stderr, n=nn, precision="mixed")
        out["mixed"]["solve_latency_s"] = {k: lat32[k] for k in ("p50_s", "p99_s", "samples")}
        out["mixed"]["solves_per_s"] = lat32["solves_per_s"]
        out["mixed"]["solve_latency_runs"] = lat32["runs"]
    if args.serve_requests > 0:
        from itofoggysim_amd import Server, poisson_workload, run_workload
        torch.cuda.synchronize()
        reqs = poisson_workload(args.serve_requests, args.serve_rate, seed=5, n_min=10, n_max=args.serve_nmax,
                                max_dirs=args.serve_dirs)
        srv = Server(slots=args.serve_slots, hbm_budget_gb=200.0)
        if args.serve_verbose:
            srv.set_verbose(True)
        t0 = time.perf_counter()
        res, stt = run_workload(srv, reqs, tol=1e-6)
        wall = time.perf_counter() - t0
        srv.close()
        ok = all(info["status"] == 0 for _, info in res)
        nsolves = sum(len(r["directions"]) for r in reqs)
        out["serving"] = {
            "workload": f"{len(reqs)} requests, Poisson arrivals at {args.serve_rate} /s, N log-uniform in "
                        f"[10, {args.serve_nmax}] (20-sphere benchmark radius law and number density), lambda "
                        f"U[400,1550] nm with n = 1.3199 + 3500 nm^2/lambda^2 + 1e-8 i, 1-{args.serve_dirs} directions, "
                        f"half plain-FP64 / half mixed, GMRES(30) to 1e-6, {args.serve_slots} slots, 200 GB budget, shortest estimated request first with aging",
            "all_ok": ok, "requests": len(reqs), "solves": nsolves, "wall_s": round(wall, 3),
            "p50_latency_s": round(float(stt["p50_s"]), 4), "p99_latency_s": round(float(stt["p99_s"]), 4),
            "requests_per_s": round(len(reqs) / wall, 4), "solves_per_s": round(nsolves / wall, 4),
            "peak_concurrent": stt["peak_concurrent"], "peak_admitted_gb": round(stt["peak_admitted_bytes"] / 2**30, 2),
            "per_request": [{"n": len(r["cluster"]["radii"]), "lambda_um": round(r["cluster"]["wavelength"], 4),
                             "ndir": len(r["directions"]), "precision": r["precision"],
                             "latency_s": round(info["latency_s"], 3), "queue_s": round(info["queue_s"], 3),
                             "footprint_gb": round(info["footprint_bytes"] / 2**30, 3)} for r, (_, info) in zip(reqs, res)]}
        print(f"# serving: {len(reqs)} requests in {wall:.1f} s, p50 {stt['p50_s']:.2f} s, p99 {stt['p99_s']:.2f} s",
              file=sys.stderr, flush=True)
    if not args.no_cpu:
        # every core of the host share this process runs on: OMP_NUM_THREADS where the host
        # sets it (the CPU share of one GPU on a shared node), else all of nproc
        threads = int(os.environ.get("OMP_NUM_THREADS") or 0) or (os.cpu_count() or 1)
        out["cpu_baseline"] = cpu_baseline(c, args.cpu_pairs, threads, affinity)
    print(json.dumps(out))


if __name__ == "__main__":
    main()
