// Serving loop: continuous batching of scattering requests on one GPU.
//
// Requests (a cluster, its parameters and 1..n incidence directions) are queued
// as they arrive.  Worker slots take the oldest queued request whose estimated HBM
// footprint fits what the admitted requests leave of the budget, so requests that
// arrive while others run are admitted as soon as a slot and memory free up.
// Every admitted request owns a context with its own HIP stream: its tables and
// Krylov state stay device-resident for the whole request, and the work of
// concurrent requests overlaps on the device.  A request's result does not depend
// on what runs beside it (no shared device state, deterministic kernels).
//
// Per request: right-hand sides T p for every direction, lock-step GMRES over the
// directions (one batched matvec per Arnoldi step), then the cross sections.
#include <algorithm>
#include <array>
#include <chrono>
#include <cmath>
#include <condition_variable>
#include <cstdio>
#include <deque>
#include <map>
#include <mutex>
#include <set>
#include <thread>
#include <unordered_map>
#include <vector>

#include "../../include/ifs.h"
#include "ifs_engine.h"
#include "ifs_leaf.h"
#include "ifs_pair.h"
#include "ifs_pw.h"
#include "ifs_tree.h"

namespace {

using clk = std::chrono::steady_clock;

struct Req {
    int64_t id = 0;
    std::vector<double> centres, radii, mrel, alpha, beta;
    std::vector<int32_t> lmax;
    ifs_params prm{};
    double tol = 1e-6;
    int restart = 30, max_iter = 1000;
    size_t footprint = 0;
    double est_s = 0.0;  // estimated device time (admission order)
    clk::time_point t_submit, t_start, t_done;
    // result
    int status = 0;
    bool done = false;
    std::vector<double> csec;  // 3 per direction
    int iterations = 0;
};

}  // namespace

struct ifs_server {
    std::mutex mu;
    std::condition_variable cv_work, cv_done;
    std::deque<int64_t> queue;
    std::map<int64_t, Req> reqs;
    std::vector<std::thread> workers;
    size_t budget = 0, admitted = 0, peak_admitted = 0;
    int slots = 1;
    int running = 0, peak_running = 0;
    int64_t next_id = 1;
    bool stop = false;
    int verbose = 0;  // progress lines on stderr: each request's GMRES steps and its completion
    clk::time_point t0;
    std::vector<double> latencies;
    int64_t completed = 0;
};

namespace {

// Device memory of a request, planned on the host before admission, and the limits its
// context is created with so that it stays inside the plan (ifs_create would otherwise
// size its workspace and table cache from the free memory of the whole device):
//   vectors    right-hand sides, iterates, the lock-step GMRES basis, compact copies;
//   pools      MLFMM multipole and local expansions of every box (octree built on the
//              host with the library's own functions: scaling, Morton keys, l_max);
//   workspace  the translation workspace (ifs_params.workspace_mb), at most a quarter
//              of a slot's share of the budget and at most 8 GiB;
//   tables     translation tables kept across matvecs (ifs_params.cache_mb) of the paths
//              that ifs_create will choose, when they fit the rest of the slot's share;
//              otherwise regenerated in every matvec;
//   fixed      per-context buffers, matrices shared by all pairs, and the workspaces beside
//              the translation workspace (generators, partial sums, row coefficients).
struct Plan {
    size_t vectors = 0, pools = 0, workspace = 0, tables = 0, fixed = 0;
    double seconds = 0.0;  // device time of one product, per right-hand side
    size_t total() const { return vectors + pools + workspace + tables + fixed; }
};

int box_L(double k, double edge, double d0, int cap) {
    const double kD = k * edge;
    int L = (int)std::ceil(kD + 1.8 * std::pow(d0, 2.0 / 3.0) * std::cbrt(kD));
    if (L < 1) L = 1;
    if (cap > 0 && L > cap) L = cap;
    return L;
}

// What the translations of a request need: tables to keep, the workspaces of all right-hand
// sides (y, z: the translation workspace, each the largest of the stages that share it), the
// buffers beside it, and the time of a product.
struct Need {
    double tables = 0.0, y = 0.0, z = 0.0, s = 0.0, gen = 0.0, fixed = 0.0, seconds = 0.0;
    void work(double a, double b) {
        y = std::max(y, a);
        z = std::max(z, b);
    }
};

// Rates of the stages in the flops counted here (per pair or class translation 21 L^3, L the larger
// order): 22650 sphere pairs of orders 10 to 18 in 0.45 ms; 56046 sampled translations of orders 97
// and 174 in 5.2 ms; P2M and L2P of 2500 spheres in 4 ms; class products of orders 400 to 800.
constexpr double kPairRate = 4e12, kPwRate = 1e13, kLeafRate = 1e13, kClassRate = 4e13;

void need_pairs(const ifs::PairSize &S, int nd, Need &N) {
    const double work = std::min(S.work * nd, ifs::pair_work_cap());
    N.tables += S.tables;
    N.work(work, 0.0);
    N.s = std::max(N.s, S.sect);
    N.fixed += S.shared() + S.lists;
    N.seconds += S.flops / kPairRate;
}

// One-by-one translations of orders Ls -> Lt, K their smaller: tables, and what they take in all.
double one_by_one(double Ls, double Lt) {
    const double K = std::min(Ls, Lt), Lm = std::max(Ls, Lt);
    return 8.0 * 2.0 * (K + 1) * (Lm + 1) * (Lm + 2) / 2.0 + 16.0 * 2.0 * (2 * K + 1) * Ls * Lt +
           16.0 * 2.0 * (2 * K + 1) * (Ls + Lt);
}

// A batch of class products: `cols` translations of degrees n0..L (n0 = 1: orders Ls -> Lt) with
// so many coaxial and Wigner tables.
void need_class(int Ls, int Lt, int n0, double cols, double ax, double d, int nd, Need &N) {
    const int K = std::min(Ls, Lt);
    const double rb = (double)ifs::rows_off(n0, K), e0 = (double)n0 * n0 - 1.0;
    const double nax = 16.0 * (double)(n0 > 1 ? ifs::ax0_size(Lt, n0) : ifs::ax_size(Lt, Ls, K));
    N.tables += nax * ax + 8.0 * (double)ifs::fold_size(std::max(Ls, Lt), K) * d;
    N.work(32.0 * std::max((double)ifs::rows_size(Ls, K) - rb, (double)Lt * (Lt + 2.0) - e0) * cols * nd,
           32.0 * ((double)ifs::rows_size(Lt, K) - rb) * cols * nd);
    N.fixed += 400.0 * cols;  // lists
    const double part = n0 > 1 ? 1.0 - std::pow((double)n0 / Lt, 3.0) : 1.0, Lm = std::max(Ls, Lt);
    N.seconds += 21.0 * Lm * Lm * Lm * part * cols / kClassRate;
}

void need_tree(const Req &r, const std::vector<int> &L, size_t ws_cap, Plan &P, Need &N) {
    using namespace ifs;
    const int ns = (int)L.size(), nd = (int)r.alpha.size();
    const double k = r.prm.k, d0 = r.prm.fmm_d0 > 0.0 ? r.prm.fmm_d0 : 6.0;
    std::vector<double> scaled;
    const tree::Scaling S = tree::scale_points(r.centres.data(), ns, scaled);
    std::vector<int64_t> u(ns), us;
    for (int i = 0; i < ns; ++i) u[i] = tree::universal_index(&scaled[3 * i], tree::kThresholdLevel);
    us = u;
    std::sort(us.begin(), us.end());
    const int s = r.prm.leaf_size > 0 ? r.prm.leaf_size : 10;
    const int lmin = 2, lmax = std::max(lmin, tree::level_max(us, s));
    const bool outgoing = r.prm.z_selector != IFS_ZSEL_BESSEL_J;
    const size_t gq_cap = (size_t)1 << 30;
    auto generator = [&](int kind, double t, int Lt, int Ls) {  // boxes that no GPU holds are not worth the count
        if (std::max(Lt, Ls) > 4096) return (double)gq_cap;
        return (double)gq_plan(kind, t, Lt, Ls, std::min(Lt, Ls), gq_cap).ws_bytes;
    };
    std::unordered_map<int64_t, std::vector<int>> members;  // of the leaf boxes
    double pools = 0.0;
    int Lup = 0;
    for (int l = lmin; l <= lmax; ++l) {
        std::vector<int64_t> b(us);
        for (auto &v : b) v >>= 3 * (tree::kThresholdLevel - l);
        b.erase(std::unique(b.begin(), b.end()), b.end());
        const int nb = (int)b.size();
        const double edge = S.D / std::ldexp(1.0, l);
        const int Lb = box_L(k, edge, d0, r.prm.fmm_lmax_cap);
        pools += 2.0 * nb * 2.0 * Lb * (Lb + 2.0) * 16.0 * nd;
        if (l > lmin) {  // M2M and L2L with the level above: eight offsets of one length and polar angle
            const double t = k * edge * std::sqrt(0.75);
            need_class(Lb, Lup, 1, nb, 1, 1, nd, N);
            need_class(Lup, Lb, 1, nb, 1, 1, nd, N);
            N.gen = std::max({N.gen, generator(1, t, Lup, Lb), generator(1, t, Lb, Lup)});
        }
        Lup = Lb;
        // M2L offsets and how many boxes have each
        std::map<std::array<int, 3>, double> off;
        {
            std::unordered_map<int64_t, char> have;
            for (int64_t v : b) have[v] = 1;
            auto coords = [l](int64_t n, int v[3]) {
                v[0] = v[1] = v[2] = 0;
                for (int i = l - 1; i >= 0; --i)
                    for (int d = 0; d < 3; ++d) v[d] = (v[d] << 1) | (int)((n >> (3 * i + 2 - d)) & 1);
            };
            for (int64_t q : b) {
                int vt[3], vs[3];
                coords(q, vt);
                for (int64_t p : tree::domain_i4(q, l, 1)) {
                    if (!have.count(p)) continue;
                    coords(p, vs);
                    off[{vs[0] - vt[0], vs[1] - vt[1], vs[2] - vt[2]}] += 1.0;
                }
            }
        }
        auto o2_of = [](const std::array<int, 3> &o) { return o[0] * o[0] + o[1] * o[1] + o[2] * o[2]; };
        auto waves = [&](int o2) { return pw_takes(pw_terms(k, edge, o2, Lb), Lb); };
        double cols = 0.0;
        std::set<std::array<int, 3>> canon;
        for (auto &o : off)
            if (waves(o2_of(o.first))) {
                cols += o.second;
                const int x = std::abs(o.first[0]), y = std::abs(o.first[1]);
                canon.insert({std::max(x, y), std::min(x, y), std::abs(o.first[2])});
            }
        const bool pw = outgoing && pw_fits(ws_cap, Lb, nb, 1) && pw_worth(Lb, nb, (int64_t)cols);
        if (pw) {
            const PwSize Z = pw_size(Lb, nb * nd, Lb + 1, 2 * Lb + 0.5, 2 * Lb, Lb);
            const double nc = (double)canon.size();
            N.tables += Z.U + Z.T * nc * (r.prm.precision == IFS_PREC_MIXED ? 1.5 : 1.0);
            N.work(std::max(Z.y, 0.5 * 64.0 * 4.0 * Lb * (Lb + 2.0) * nb * nd), Z.z);
            N.fixed += 16.0 * nc * (2.0 * Lb + 1.0) + 16.0 * cols;
            N.seconds += (Z.box_flops * nb + 16.0 * Z.samples * cols) / kPwRate;
        }
        // class products: whole offsets, and the last degrees of near ones, one batch a length
        std::map<int, std::pair<double, std::set<double>>> rem;
        std::set<int> ax;
        std::set<double> d;
        double whole = 0.0;
        for (auto &o : off) {
            const int o2 = o2_of(o.first);
            const int terms = pw_terms(k, edge, o2, Lb);
            const double cth = std::fabs(o.first[2] / std::sqrt((double)o2));
            if (pw && waves(o2)) {
                if (terms >= 2 * Lb) continue;
                rem[o2].first += o.second;
                rem[o2].second.insert(cth);
            } else {
                whole += o.second;
                ax.insert(o2);
                d.insert(cth);
            }
        }
        for (auto &q : rem) {
            const int lo = pw_terms(k, edge, q.first, Lb) + 1;
            need_class(Lb, Lb, lo - Lb, q.second.first, 1, (double)q.second.second.size(), nd, N);
            N.gen = std::max(N.gen, (double)gq_plan_rem(k * edge * std::sqrt((double)q.first), Lb, lo, gq_cap).ws_bytes);
        }
        if (whole > 0.0) {
            need_class(Lb, Lb, 1, whole, (double)ax.size(), (double)d.size(), nd, N);
            N.gen = std::max(N.gen, generator(outgoing ? IFS_ZSEL_HANKEL1 : IFS_ZSEL_BESSEL_J,
                                              k * edge * std::sqrt((double)*ax.rbegin()), Lb, Lb));
        }
        if (l < lmax) continue;
        // spheres and their leaf boxes
        LeafReach R;
        double batch = 0.0;
        for (int i = 0; i < ns; ++i) {
            const int64_t q = u[i] >> (3 * (tree::kThresholdLevel - l));
            members[q].push_back(i);
            double c[3], t2 = 0.0;
            tree::centre(q, l, c);
            for (int e = 0; e < 3; ++e) {
                const double v = r.centres[3 * i + e] - (c[e] * S.D + S.x_min[e]);
                t2 += v * v;
            }
            R.add(L[i], k * std::sqrt(t2));
            batch += 2.0 * (one_by_one(L[i], Lb) + 64.0 * Lb * (2.0 * L[i] + 1.0));
        }
        if (leaf_worth(ws_cap, R, Lb, nb, ns)) {
            const PwSize Z = pw_size(Lb, nb * nd, R.nodes(Lb), R.t, R.deg(), R.order);
            N.tables += Z.U;
            N.work(Z.y, Z.z);
            N.fixed += 16.0 * R.nodes(Lb) * (R.order + 1.0) * (R.order + 2.0) / 2.0 + 200.0 * ns;
            N.s = std::max(N.s, std::min((double)ws_cap / 8.0, 64.0 * R.nodes(Lb) * (2.0 * R.order + 1.0) * ns * nd));
            N.seconds += Z.box_flops * nb / kPwRate;
            for (int i = 0; i < ns; ++i) N.seconds += 2.0 * (8.0 * L[i] + 150.0) * Z.samples / kLeafRate;
        } else {
            N.s = std::max(N.s, std::min(batch, (double)ws_cap));  // in buffers of its own
            N.gen = std::max(N.gen, (R.order + 1.0) * (Lb + 2.0) * (Lb + R.order + R.deg()) * 4.0);
            for (int i = 0; i < ns; ++i) N.seconds += 2.0 * 21.0 * L[i] * (double)Lb * Lb / kPairRate;
        }
    }
    P.pools = (size_t)pools;
    // near field; of many spheres every so-manieth stands for the others
    PairSize Q;
    double generic = 0.0;
    const int step = std::max(1, ns / 2048);
    bool takes = outgoing && *std::max_element(L.begin(), L.end()) <= kPairMaxL;
    std::vector<Task> tasks;
    for (int j = 0; j < ns; j += step) {
        tasks.clear();
        for (int64_t b : tree::domain_i2(u[j] >> (3 * (tree::kThresholdLevel - lmax)), lmax, 1)) {
            auto it = members.find(b);
            if (it == members.end()) continue;
            for (int i : it->second) {
                if (i == j) continue;
                double dv[3];
                for (int d = 0; d < 3; ++d) dv[d] = r.centres[3 * j + d] - r.centres[3 * i + d];
                tasks.push_back(make_task(dv, k, IFS_ZSEL_HANKEL1, L[i], L[j], 0, 0));
                generic += step * one_by_one(L[i], L[j]);
                takes = takes && tasks.back().t > 0.0;
            }
        }
        if (takes) pair_size(tasks, step, Q);
    }
    if (takes) {
        need_pairs(Q, nd, N);
    } else {
        N.tables += generic;
        N.s = std::max(N.s, std::min(generic, (double)ws_cap));
        N.seconds += generic / 1e12;
    }
}

void need_direct(const Req &r, const std::vector<int> &L, Need &N) {
    using namespace ifs;
    const int ns = (int)L.size(), nd = (int)r.alpha.size();
    bool takes = r.prm.z_selector != IFS_ZSEL_BESSEL_J && *std::max_element(L.begin(), L.end()) <= kPairMaxL;
    PairSize Q;
    std::vector<Task> tasks;
    // of many spheres every so-manieth stands for the others
    const int step = std::max(1, ns / 512);
    for (int j = 0; j < ns && takes; j += step) {
        tasks.clear();
        for (int i = 0; i < ns; ++i) {
            if (i == j) continue;
            double dv[3];
            for (int d = 0; d < 3; ++d) dv[d] = r.centres[3 * j + d] - r.centres[3 * i + d];
            tasks.push_back(make_task(dv, r.prm.k, IFS_ZSEL_HANKEL1, L[i], L[j], 0, 0));
            takes = takes && tasks.back().t > 0.0;
        }
        pair_size(tasks, (double)step, Q);
    }
    if (takes) {
        need_pairs(Q, nd, N);
        return;
    }
    double t = 0.0;
    for (int a = 0; a < ns; ++a)
        for (int b = 0; b < ns; ++b)
            if (a != b) t += one_by_one(L[a], L[b]);
    N.tables += t;
    N.work(t * nd, 0.0);
    N.seconds += t / 1e12;
}

Plan plan_request(Req &r, size_t budget, int slots) {
    Plan P;
    const int ns = (int)r.radii.size();
    int N = r.prm.n_global;
    const double k = r.prm.k;
    std::vector<int> L(ns);
    for (int j = 0; j < ns; ++j) {
        int lj = r.lmax.empty() ? (int)std::ceil(k * r.radii[j] + 4.05 * std::cbrt(k * r.radii[j]) + 2.0) : r.lmax[j];
        L[j] = std::max(1, N > 0 ? std::min(lj, N) : lj);
    }
    if (N <= 0) N = *std::max_element(L.begin(), L.end());
    const double n = 2.0 * ns * N * (N + 2);
    const int nd = (int)r.alpha.size();
    P.vectors = (size_t)(16.0 * n * ((r.restart + 1) * nd + 6.0 * nd + 4.0));
    const size_t share = budget / (size_t)std::max(slots, 1);
    const size_t ws_cap = std::min<size_t>(std::max<size_t>(share / 4, (size_t)256 << 20), (size_t)8 << 30);
    Need D;
    if (r.prm.use_fmm)
        need_tree(r, L, ws_cap, P, D);
    else
        need_direct(r, L, D);
    P.seconds = D.seconds;
    P.workspace = (size_t)std::min<double>((double)ws_cap, D.y + D.z + (64 << 20));
    // counted rather than planned: a tenth more, and the per-context buffers.  Wigner tables
    // regenerated in a product take at most a quarter of the workspace.
    P.fixed = (size_t)(1.1 * (D.s + D.gen + D.fixed)) + ((size_t)96 << 20);
    const double table_need = 1.1 * D.tables;
    // tables kept only when they fit what the slot's share leaves
    const size_t used = P.vectors + P.pools + P.workspace + P.fixed;
    if (table_need > 0.0 && (double)used + table_need <= (double)share)
        P.tables = (size_t)table_need;
    else if (r.prm.use_fmm)
        P.fixed += P.workspace / 4;
    r.prm.workspace_mb = (int32_t)std::max<size_t>(1, P.workspace >> 20);
    r.prm.cache_mb = P.tables > 0 ? (int32_t)((P.tables >> 20) + 1) : -1;
    if (P.tables > 0) P.tables = (size_t)r.prm.cache_mb << 20;
    return P;
}

void run_request(Req &r, int verbose) {
    ifs_cluster cl{(int32_t)r.radii.size(), r.centres.data(), r.radii.data(), r.mrel.data(),
                   r.lmax.empty() ? nullptr : r.lmax.data()};
    ifs_ctx *c = nullptr;
    int rc = ifs_create(&c, &cl, &r.prm);
    if (rc) {
        r.status = rc;
        return;
    }
    const int nd = (int)r.alpha.size();
    const int64_t n = ifs_vector_length(c);
    std::vector<double> rhs(2 * n * nd), p(2 * n * nd), x(2 * n * nd);
    for (int d = 0; d < nd && !rc; ++d) {
        rc = ifs_plane_wave_rhs_dir(c, r.alpha[d], r.beta[d], rhs.data() + 2 * n * d, n);
        if (!rc) rc = ifs_plane_wave(c, r.alpha[d], r.beta[d], p.data() + 2 * n * d, n);
    }
    std::vector<ifs_solve_info> info(nd);
    if (!rc) {
        ifs_solve_opts op{r.restart, r.max_iter, r.tol, 0, verbose, r.prm.precision, 0};
        rc = ifs_solve_batch(c, nd, rhs.data(), x.data(), n, &op, info.data());
    }
    r.csec.assign(3 * nd, 0.0);
    for (int d = 0; d < nd && (rc == IFS_OK || rc == IFS_E_NOCONV); ++d) {
        int q = ifs_cross_sections(c, x.data() + 2 * n * d, p.data() + 2 * n * d, n, r.csec.data() + 3 * d);
        if (q) rc = q;
        r.iterations = std::max(r.iterations, info[d].iterations);
    }
    r.status = rc;
    ifs_destroy(c);
}

void worker(ifs_server *s) {
    std::unique_lock<std::mutex> lk(s->mu);
    for (;;) {
        // among the queued requests whose footprint fits (any one if nothing runs), the one
        // with the least estimated device time less its waiting time: short requests pass
        // long ones, and a long one's priority grows as it waits (no starvation)
        int64_t pick = 0;
        s->cv_work.wait(lk, [&] {
            if (s->stop && s->queue.empty()) return true;
            const clk::time_point now = clk::now();
            double best = 0.0;
            pick = 0;
            for (int64_t id : s->queue) {
                Req &r = s->reqs[id];
                if (!(s->admitted + r.footprint <= s->budget || s->running == 0)) continue;
                const double prio = r.est_s - std::chrono::duration<double>(now - r.t_submit).count();
                if (!pick || prio < best) {
                    pick = id;
                    best = prio;
                }
            }
            return pick != 0;
        });
        if (!pick) {
            if (s->stop && s->queue.empty()) return;
            continue;
        }
        s->queue.erase(std::find(s->queue.begin(), s->queue.end(), pick));
        Req &r = s->reqs[pick];
        s->admitted += r.footprint;
        s->peak_admitted = std::max(s->peak_admitted, s->admitted);
        s->running += 1;
        s->peak_running = std::max(s->peak_running, s->running);
        r.t_start = clk::now();
        const int verbose = s->verbose;
        lk.unlock();
        run_request(r, verbose);  // r stays valid: map nodes are stable and erased only by the waiter
        lk.lock();
        r.t_done = clk::now();
        if (verbose) {
            std::fprintf(stderr, "serve: request %lld done: %zu spheres, %zu directions, %s, %.1f s (queued %.1f s), "
                                 "status %d\n",
                         (long long)r.id, r.radii.size(), r.alpha.size(),
                         r.prm.precision == IFS_PREC_MIXED ? "mixed" : "fp64",
                         std::chrono::duration<double>(r.t_done - r.t_submit).count(),
                         std::chrono::duration<double>(r.t_start - r.t_submit).count(), r.status);
            std::fflush(stderr);
        }
        r.done = true;
        s->admitted -= r.footprint;
        s->running -= 1;
        s->latencies.push_back(std::chrono::duration<double>(r.t_done - r.t_submit).count());
        s->completed += 1;
        s->cv_done.notify_all();
        s->cv_work.notify_all();
    }
}

}  // namespace

extern "C" {

int ifs_server_set_verbose(ifs_server *s, int32_t verbose) {
    if (!s || (verbose != 0 && verbose != 1)) return IFS_E_ARG;
    std::lock_guard<std::mutex> lk(s->mu);
    s->verbose = verbose;
    return IFS_OK;
}

int ifs_server_create(ifs_server **out, int32_t slots, double hbm_budget_gb) {
    if (!out || slots < 1 || slots > 64 || !(hbm_budget_gb > 0.0)) return IFS_E_ARG;
    ifs_server *s = new ifs_server();
    s->budget = (size_t)(hbm_budget_gb * 1073741824.0);
    s->slots = slots;
    s->t0 = clk::now();
    for (int i = 0; i < slots; ++i) s->workers.emplace_back(worker, s);
    *out = s;
    return IFS_OK;
}

int ifs_server_submit(ifs_server *s, const ifs_cluster *cl, const ifs_params *prm, int32_t ndir, const double *alpha,
                      const double *beta, double tol, int32_t restart, int64_t *id_out) {
    if (!s || !cl || !prm || ndir < 1 || !alpha || !beta || !id_out || cl->n_spheres < 1 || !cl->centres ||
        !cl->radii || !cl->m_rel || !(tol > 0.0) || restart < 1)
        return IFS_E_ARG;
    Req r;
    const int ns = cl->n_spheres;
    r.centres.assign(cl->centres, cl->centres + 3 * ns);
    r.radii.assign(cl->radii, cl->radii + ns);
    r.mrel.assign(cl->m_rel, cl->m_rel + 2 * ns);
    if (cl->lmax) r.lmax.assign(cl->lmax, cl->lmax + ns);
    r.alpha.assign(alpha, alpha + ndir);
    r.beta.assign(beta, beta + ndir);
    r.prm = *prm;
    r.tol = tol;
    r.restart = restart;
    if (r.prm.precision != IFS_PREC_FP64 && r.prm.precision != IFS_PREC_MIXED) return IFS_E_ARG;
    // the context's workspace and table cache come from the plan, not from free memory
    {
        const Plan P = plan_request(r, s->budget, s->slots);
        r.footprint = P.total();
        r.est_s = 20.0 * P.seconds * (double)r.alpha.size();  // about 20 products a solve
    }
    std::lock_guard<std::mutex> lk(s->mu);
    if (s->stop) return IFS_E_ARG;
    r.id = s->next_id++;
    r.t_submit = clk::now();
    *id_out = r.id;
    s->reqs.emplace(r.id, std::move(r));
    s->queue.push_back(*id_out);
    s->cv_work.notify_all();
    return IFS_OK;
}

int ifs_server_plan(const ifs_cluster *cl, const ifs_params *prm, int32_t ndir, int32_t restart,
                    double hbm_budget_gb, int32_t slots, double out[8]) {
    if (!cl || !prm || !out || ndir < 1 || cl->n_spheres < 1 || !cl->centres || !cl->radii || restart < 1 ||
        slots < 1 || !(hbm_budget_gb > 0.0))
        return IFS_E_ARG;
    Req r;
    const int ns = cl->n_spheres;
    r.centres.assign(cl->centres, cl->centres + 3 * ns);
    r.radii.assign(cl->radii, cl->radii + ns);
    if (cl->lmax) r.lmax.assign(cl->lmax, cl->lmax + ns);
    r.alpha.assign((size_t)ndir, 0.0);
    r.beta.assign((size_t)ndir, 0.0);
    r.prm = *prm;
    r.restart = restart;
    const Plan P = plan_request(r, (size_t)(hbm_budget_gb * 1073741824.0), slots);
    out[0] = (double)P.vectors;
    out[1] = (double)P.pools;
    out[2] = (double)P.workspace;
    out[3] = (double)P.tables;
    out[4] = (double)P.fixed;
    out[5] = (double)P.total();
    out[6] = (double)r.prm.workspace_mb;
    out[7] = (double)r.prm.cache_mb;
    return IFS_OK;
}

int ifs_server_wait(ifs_server *s, int64_t id, double *csec, ifs_request_info *info) {
    if (!s) return IFS_E_ARG;
    std::unique_lock<std::mutex> lk(s->mu);
    auto it = s->reqs.find(id);
    if (it == s->reqs.end()) return IFS_E_ARG;
    s->cv_done.wait(lk, [&] { return it->second.done; });
    Req &r = it->second;
    if (csec) std::copy(r.csec.begin(), r.csec.end(), csec);
    if (info) {
        info->status = r.status;
        info->iterations = r.iterations;
        info->latency_s = std::chrono::duration<double>(r.t_done - r.t_submit).count();
        info->queue_s = std::chrono::duration<double>(r.t_start - r.t_submit).count();
        info->footprint_bytes = (int64_t)r.footprint;
    }
    int st = r.status;
    s->reqs.erase(it);
    return st;
}

int ifs_server_stats(ifs_server *s, double out[6]) {
    if (!s || !out) return IFS_E_ARG;
    std::lock_guard<std::mutex> lk(s->mu);
    std::vector<double> l = s->latencies;
    std::sort(l.begin(), l.end());
    auto pct = [&](double q) {
        if (l.empty()) return 0.0;
        size_t i = (size_t)std::ceil(q * l.size()) - 1;
        return l[std::min(i, l.size() - 1)];
    };
    double el = std::chrono::duration<double>(clk::now() - s->t0).count();
    out[0] = (double)s->completed;
    out[1] = pct(0.50);
    out[2] = pct(0.99);
    out[3] = el > 0.0 ? s->completed / el : 0.0;
    out[4] = (double)s->peak_running;
    out[5] = (double)s->peak_admitted;
    return IFS_OK;
}

int ifs_server_destroy(ifs_server *s) {
    if (!s) return IFS_OK;
    {
        std::lock_guard<std::mutex> lk(s->mu);
        s->stop = true;
        s->cv_work.notify_all();
    }
    for (auto &t : s->workers) t.join();
    delete s;
    return IFS_OK;
}

}  // extern "C"
