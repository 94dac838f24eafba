// Plan and launch order of the sampled P2M and L2P (kernels: ifs_leaf.hip).
#include "ifs_leaf.h"

#include <algorithm>
#include <cmath>

namespace ifs {

namespace {

int upload(DevBuf &d, const void *h, size_t bytes) {
    int rc = d.alloc(std::max<size_t>(bytes, 16));
    if (rc) return rc;
    if (bytes && hipMemcpy(d.p, h, bytes, hipMemcpyHostToDevice) != hipSuccess) return IFS_E_HIP;
    return IFS_OK;
}

// Translation vector of a task (k |d|, its direction) turned by pi about z: the exponent's.
void exponent(const Task &T, double v[3]) {
    const double st = std::sqrt(std::max(0.0, (1.0 - T.cth) * (1.0 + T.cth)));
    v[0] = -T.t * st * std::cos(T.phi);
    v[1] = -T.t * st * std::sin(T.phi);
    v[2] = T.t * T.cth;
}

// Coefficients of all rows of one sphere and right-hand side (complex).
int64_t row_coefs(const Leaf &F) { return 2LL * F.g.Q2 * 2 * (2 * F.Nmax + 1); }

// Algorithmic flops of spheres s0 .. s0 + n - 1 and one right-hand side: on a chunk's samples
// (8 N + 150 a sample) with their row sums (P2M), and of the sums over all rows (L2P).
double sample_flops(const std::vector<LeafSphere> &v, int s0, int n, const PwLevel::Chunk &ch, bool rows) {
    double f = 0.0;
    for (int i = s0; i < s0 + n; ++i)
        f += (8.0 * v[i].N + 150.0) * (double)ch.sn + (rows ? 16.0 * ch.R2 * v[i].N * (v[i].N + 2.0) : 0.0);
    return f;
}
double sum_flops(const std::vector<LeafSphere> &v, int s0, int n, int Q2) {
    double f = 0.0;
    for (int i = s0; i < s0 + n; ++i) f += 16.0 * Q2 * v[i].N * (v[i].N + 2.0);
    return f;
}

LeafArg leaf_arg(ifs_ctx *c, Leaf &F, int nrhs) {
    LeafArg a{};
    a.p = pw_arg(c, F.g, nrhs);
    a.mu = F.g.d_mu.as<double>();
    a.us = F.d_us.as<double>();
    a.ucols = (F.Nmax + 1) * (F.Nmax + 2) / 2;
    a.nb = F.g.nb;
    a.Nmax = F.Nmax;
    return a;
}

// The box matrices of a chunk's rows: kept for all rows, or made in the workspace.
void box_matrices(ifs_ctx *c, Leaf &F, LeafArg &a, const PwLevel::Chunk &ch, size_t i) {
    PwLevel &P = F.g;
    a.p.j0 = ch.j0;
    a.p.R2 = ch.R2;
    a.p.cpre = P.d_cpre.as<int64_t>() + P.cpre_at[i];
    double *U = P.kept ? P.own_U.as<double>() : c->ws_d.as<double>();
    a.p.U = U;
    if (P.kept) {
        a.p.ustr = 2 * P.Q2;
        if (!P.ready) {
            Scope s(c, "leaf_gen_tables");
            launch_pw_utable(P.L, P.Q2, 0, P.Q2, 0, P.Q2, a.p.ustr, a.mu, U, c->stream);
            P.ready = !capturing(c);
        }
        a.p.a0 = ch.j0;
        a.p.a1 = P.Q2 + ch.j0;
    } else {
        a.p.ustr = 2 * ch.R2;
        a.p.a0 = 0;
        a.p.a1 = ch.R2;
        Scope s(c, "leaf_gen_tables");
        launch_pw_utable(P.L, P.Q2, ch.j0, ch.R2, 0, ch.R2, a.p.ustr, a.mu, U, c->stream);
    }
}

}  // namespace

// The synthesis and analysis of a box cost about what one sphere of order 20 does one by one
// (order 410: 50 us against 55 us), so from 1.5 spheres a box on; below order 32 both are
// launches.
bool leaf_worth(size_t ws_budget, const LeafReach &R, int L, int nb, int ns) {
    if (L < 32 || L > 850 || 2 * ns < 3 * nb || !pw_fits(ws_budget, L, nb, 1)) return false;
    // what the blocks hold in LDS: sphere orders up to 511, and rows of up to 1984 azimuths (box order,
    // sphere order and the factor's degree together; 2 L + 250 where the spheres are small)
    const int maxN = pw_max_azimuths(L, R.t, R.deg(), R.order);
    return leaf_p2m_lds(R.order) <= 65536 && leaf_l2p_lds(maxN) <= 65536 && maxN <= kPwMaxN;
}

int LeafReach::deg() const { return (int)std::ceil(t + 8.0 * std::cbrt(t) + 30.0); }

int LeafReach::nodes(int L) const { return (L + order + deg()) / 4 + 1; }

LeafReach leaf_reach(const std::vector<Task> &p2m, const std::vector<Task> &l2p) {
    LeafReach R;
    for (auto &T : p2m) R.add(T.Ls, T.t);
    for (auto &T : l2p) R.add(T.Lt, T.t);
    return R;
}

int leaf_prepare(ifs_ctx *c, Leaf &F, int nrhs) {
    const int g = pw_group(c, F.g, nrhs);
    if (F.g.plan_nrhs != g) {
        if (hipStreamSynchronize(c->stream) != hipSuccess) return IFS_E_HIP;
        // row coefficients of the spheres: an eighth of the workspace, at least one sphere
        const int64_t per = row_coefs(F) * g;
        F.gcap = std::max<int64_t>(1, std::min<int64_t>((int64_t)std::max(F.up.size(), F.down.size()),
                                                        (int64_t)(c->ws_budget / 8 / 16) / per));
        F.g.ws.s = 16 * (size_t)(F.gcap * per);
        int rc = pw_plan(c, F.g, g);
        if (rc) return rc;
    }
    return ws_reserve(c, F.g.ws);
}

int leaf_build(ifs_ctx *c, Leaf &F, const std::vector<Task> &p2m, const std::vector<Task> &l2p, int L, int nb,
               int64_t off) {
    PwLevel &P = F.g;
    P.L = L;
    P.nb = nb;
    P.off = off;
    const int64_t per_box = 2LL * L * (L + 2);
    const LeafReach R = leaf_reach(p2m, l2p);
    F.Nmax = R.order;
    F.first.assign(nb + 1, 0);
    for (auto &T : p2m) {
        LeafSphere S{T.src, T.Ls, (int32_t)((T.dst - off) / per_box), {0, 0, 0}};
        exponent(T, S.v);
        F.up.push_back(S);
        ++F.first[S.box + 1];
    }
    for (int b = 0; b < nb; ++b) F.first[b + 1] += F.first[b];
    for (auto &T : l2p) {
        LeafSphere S{T.dst, T.Lt, (int32_t)((T.src - off) / per_box), {0, 0, 0}};
        exponent(T, S.v);
        F.down.push_back(S);
    }
    std::stable_sort(F.up.begin(), F.up.end(), [](auto &a, auto &b) { return a.box < b.box; });
    std::stable_sort(F.down.begin(), F.down.end(), [](auto &a, auto &b) { return a.box < b.box; });
    int rc = pw_grid(c, P, R.nodes(L), R.t, R.deg(), F.Nmax);
    if (rc) return rc;
    const int ucols = (F.Nmax + 1) * (F.Nmax + 2) / 2;
    if ((rc = upload(F.d_up, F.up.data(), sizeof(LeafSphere) * F.up.size())) ||
        (rc = upload(F.d_down, F.down.data(), sizeof(LeafSphere) * F.down.size())) ||
        (rc = upload(F.d_first, F.first.data(), 4 * F.first.size())) ||
        (rc = F.d_us.alloc(16 * (size_t)P.Q2 * ucols)))
        return rc;
    launch_leaf_utable(F.Nmax, P.Q2, ucols, P.d_mu.as<double>(), F.d_us.as<double>(), c->stream);
    const size_t ub = 8 * (size_t)pw_ucnt(L + 1, L) * 2 * P.Q2;
    P.kept = ub + c->ws_cached <= c->cache_budget && P.own_U.alloc(ub) == IFS_OK;
    if (P.kept)
        c->ws_cached += ub;
    else
        (void)hipGetLastError();
    if (hipPeekAtLastError() != hipSuccess) return IFS_E_HIP;
    return leaf_prepare(c, F, 1);
}

int leaf_p2m(ifs_ctx *c, Leaf &F, const double2 *xh, double2 *C, int nrhs, int64_t ldx, int64_t ldC) {
    const int g = pw_group(c, F.g, nrhs);
    if (int rc = leaf_prepare(c, F, nrhs)) return rc;
    for (int r0 = 0; r0 < nrhs; r0 += g) {
        const int nr = std::min(g, nrhs - r0);
        LeafArg a = leaf_arg(c, F, nr);
        double2 *rows = c->ws_s.as<double2>();
        const int ns = (int)F.up.size();
        for (size_t i = 0; i < F.g.chunks.size(); ++i) {
            const auto &ch = F.g.chunks[i];
            box_matrices(c, F, a, ch, i);
            {
                Scope s(c, "p2m_samples", sample_flops(F.up, 0, ns, ch, true) * nr);
                for (int s0 = 0; s0 == 0 || s0 < ns; s0 += (int)F.gcap)
                    launch_leaf_p2m(a, F.d_up.as<LeafSphere>(), F.d_first.as<int32_t>(), s0,
                                    std::min<int>((int)F.gcap, ns - s0), xh + r0 * ldx, ldx, nr, ch.maxN, rows, s0 > 0,
                                    c->stream);
            }
            Scope s(c, "p2m_box", (ch.f_fft + ch.f_gemm) * F.g.nb * nr);
            launch_pw_fft(a.p, 1, ch.maxN, c->stream);
            launch_pw_anal(a.p, i > 0, c->stream);
        }
        Scope s(c, "p2m_box");
        launch_pw_unpack(a.p, F.g.nb, F.g.off, C + r0 * ldC, ldC, c->stream);
    }
    return hipPeekAtLastError() == hipSuccess ? IFS_OK : IFS_E_HIP;
}

int leaf_l2p(ifs_ctx *c, Leaf &F, const double2 *D, double2 *acc, int nrhs, int64_t ldD, int64_t ldacc) {
    const int g = pw_group(c, F.g, nrhs);
    if (int rc = leaf_prepare(c, F, nrhs)) return rc;
    for (int r0 = 0; r0 < nrhs; r0 += g) {
        const int nr = std::min(g, nrhs - r0);
        LeafArg a = leaf_arg(c, F, nr);
        double2 *rows = c->ws_s.as<double2>();
        const int ns = (int)F.down.size();
        // every sphere group needs the samples of all rows: with one chunk they are made once
        for (int s0 = 0; s0 < ns; s0 += (int)F.gcap) {
            const int n = std::min<int>((int)F.gcap, ns - s0);
            const bool made = F.g.chunks.size() == 1 && s0 > 0;
            if (!made) {
                Scope s(c, "l2p_box");
                launch_pw_pack(a.p, F.g.nb, F.g.off, D + r0 * ldD, ldD, c->stream);
            }
            for (size_t i = 0; i < F.g.chunks.size(); ++i) {
                const auto &ch = F.g.chunks[i];
                box_matrices(c, F, a, ch, i);
                if (!made) {
                    Scope s(c, "l2p_box", (ch.f_fft + ch.f_gemm) * F.g.nb * nr);
                    launch_pw_synth(a.p, c->stream);
                    launch_pw_fft(a.p, 0, ch.maxN, c->stream);
                }
                Scope s(c, "l2p_samples", sample_flops(F.down, s0, n, ch, false) * nr);
                launch_leaf_l2p(a, F.d_down.as<LeafSphere>(), s0, n, nr, ch.maxN, rows, c->stream);
            }
            Scope s(c, "l2p_sum", sum_flops(F.down, s0, n, F.g.Q2) * nr);
            launch_leaf_sum(a, F.d_down.as<LeafSphere>(), s0, n, nr, rows, acc + r0 * ldacc, ldacc, c->stream);
        }
    }
    return hipPeekAtLastError() == hipSuccess ? IFS_OK : IFS_E_HIP;
}

uint64_t leaf_sig(const Leaf &F) {
    uint64_t h = pw_sig(F.g);
    for (const DevBuf *d : {&F.d_up, &F.d_down, &F.d_first, &F.d_us})
        h ^= (uint64_t)(uintptr_t)d->p + 0x9e3779b97f4a7c15ull + (h << 6) + (h >> 2);
    return h;
}

}  // namespace ifs
