// Plan and launch order of the plane-wave M2L (kernels: ifs_pw.hip).
#include "ifs_pw.h"

#include <algorithm>
#include <cmath>
#include <map>

namespace ifs {

namespace {

int upload(DevBuf &d, const void *h, size_t bytes) {
    int rc = d.alloc(std::max<size_t>(bytes, 16));
    if (rc) return rc;
    if (bytes && hipMemcpy(d.p, h, bytes, hipMemcpyHostToDevice) != hipSuccess) return IFS_E_HIP;
    return IFS_OK;
}

// Smallest multiple of 4 that is >= n and has no prime factor above 5.
int fft_length(int n) {
    for (int m = (n + 3) / 4 * 4;; m += 4) {
        int r = m;
        for (int p : {2, 3, 5})
            while (r % p == 0) r /= p;
        if (r == 1) return m;
    }
}

PwFft fft_plan(int N, std::vector<double2> &tw, std::vector<int32_t> &perm) {
    PwFft F{};
    F.N = N;
    int r = N;
    auto take = [&](int q) {
        while (r % q == 0) {
            F.radix[F.npass++] = q;
            r /= q;
        }
    };
    take(4);
    take(2);
    take(3);
    take(5);
    F.tw = (int)tw.size();
    F.perm = (int)perm.size();
    for (int i = 0; i < N; ++i) {
        const long double a = 2.0L * 3.14159265358979323846264338327950288L * i / N;
        tw.push_back(make_double2((double)cosl(a), (double)sinl(a)));
    }
    // position sum q_i N/(r_1..r_i) holds frequency q_1 + r_1 q_2 + r_1 r_2 q_3 + ...
    for (int k = 0; k < N; ++k) {
        int pos = 0, rest = k, len = N;
        for (int i = 0; i < F.npass; ++i) {
            len /= F.radix[i];
            pos += (rest % F.radix[i]) * len;
            rest /= F.radix[i];
        }
        perm.push_back(pos);
    }
    return F;
}

// Largest order of a function of degree nu that reaches 1e-16 at polar angle asin(s):
// there U falls at least like J_m(nu s), and (m - x)/(x/2)^{1/3} = 14.5 is 1e-16.
int m_reach(double nu, double s, int cap) {
    const double x = nu * s;
    return std::min(cap, (int)std::ceil(x + 11.5 * std::cbrt(x) + 10.0));
}

int64_t x_size(int L) { return 2 * (pw_xcnt(L, L) + pw_cn(L, L)); }

}  // namespace

int pw_terms(double k, double edge, int o2, int L) {
    const double t = k * edge * std::sqrt((double)o2);
    return std::min(2 * L, (int)(t + 2.5 * std::cbrt(0.5 * t)));
}

// A box costs about 1.5 class translations and some ten launches; measured M2L time with
// and without: order 34, 42 translations a box 0.98 against 3.3 ms, order 60, 22 a box 0.61
// against 3.2 ms, order 78, 48 a box 1.2 against 13.7 ms.  Below 16 a box (trees of a few
// dozen spheres) or order 32 both are launches, and the class products stay.
bool pw_worth(int L, int nb, int64_t cols) { return L >= 32 && cols >= 16LL * nb; }

bool pw_fits(size_t ws_budget, int L, int nb, int nrhs) {
    return 4 * L + 1 <= kPwMaxN - 96 && 64.0 * (double)x_size(L) * nb * nrhs <= (double)ws_budget;
}

int pw_group(ifs_ctx *c, const PwLevel &P, int nrhs) {
    while (nrhs > 1 && !pw_fits(c->ws_budget, P.L, P.nb, nrhs)) --nrhs;
    return nrhs;
}

namespace {
// Azimuths of a row at polar angle asin(s) whose transform keeps the orders up to mF.
int azimuths(int mF, double s, double tdeg, int tcap, int order) {
    const int N = fft_length(mF + m_reach(order + 0.5, s, order) + m_reach(tdeg, s, tcap) + 1);
    return N < 2 * mF + 1 ? fft_length(2 * mF + 1) : N;  // the transform reads every order up to mF
}
}  // namespace

int pw_max_azimuths(int L, double tdeg, int tcap, int order) {
    return azimuths(m_reach(L + 0.5, 1.0, L), 1.0, tdeg, tcap, order);
}

PwSize pw_size(int L, int nbr, int Q2, double tdeg, int tcap, int order) {
    PwSize S;
    for (int j = 0; j < Q2; ++j) {
        // the j-th node of the rule of 2 Q2 nodes, to about 1 / (8 Q2)^2
        const double s = std::sin(3.14159265358979323846 * (4.0 * j + 3.0) / (8.0 * Q2 + 2.0));
        const int mF = m_reach(L + 0.5, s, L), N = azimuths(mF, s, tdeg, tcap, order);
        S.samples += 2.0 * N;
        double gemm, fft;
        pw_row_flops(L, mF, N, gemm, fft);
        S.box_flops += 2.0 * (gemm + fft);
    }
    S.U = 8.0 * (double)pw_ucnt(L + 1, L) * 2.0 * Q2;
    S.T = 16.0 * S.samples;
    S.y = 16.0 * (2.0 * (double)x_size(L) + 4.0 * (2.0 * L + 1.0) * Q2) * nbr;
    S.z = 64.0 * S.samples * nbr;
    return S;
}

int pw_grid(ifs_ctx *c, PwLevel &P, int Q2, double tdeg, int tcap, int order) {
    const int L = P.L;
    P.Q2 = Q2;
    std::vector<double> x, w;
    gauss_legendre(2 * P.Q2, x, w);
    std::vector<double> mu(2 * P.Q2);
    std::vector<double2> tw;
    std::vector<int32_t> perm;
    std::map<int, int> lens;
    P.N.resize(P.Q2);
    P.mF.resize(P.Q2);
    P.fft_of.resize(P.Q2);
    for (int j = 0; j < P.Q2; ++j) {
        mu[j] = -x[j];  // from the north pole to the equator
        mu[P.Q2 + j] = w[j];
        const double s = std::sqrt((1.0 - mu[j]) * (1.0 + mu[j]));
        P.mF[j] = m_reach(L + 0.5, s, L);
        P.N[j] = azimuths(P.mF[j], s, tdeg, tcap, order);
        auto it = lens.find(P.N[j]);
        if (it == lens.end()) {
            it = lens.emplace(P.N[j], (int)P.fft.size()).first;
            P.fft.push_back(fft_plan(P.N[j], tw, perm));
        }
        P.fft_of[j] = it->second;
    }
    P.jlo.resize(L + 1);
    for (int m = 0, j = 0; m <= L; ++m) {
        while (P.mF[j] < m) ++j;
        P.jlo[m] = j;
    }
    std::vector<int64_t> gpre(2 * P.Q2);
    P.SN = 0;
    for (int t = 0; t < 2 * P.Q2; ++t) {
        gpre[t] = P.SN;
        P.SN += P.N[t % P.Q2];
    }
    int rc;
    if ((rc = upload(P.d_mu, mu.data(), 8 * mu.size())) || (rc = upload(P.d_N, P.N.data(), 4 * P.N.size())) ||
        (rc = upload(P.d_mF, P.mF.data(), 4 * P.mF.size())) || (rc = upload(P.d_jlo, P.jlo.data(), 4 * P.jlo.size())) ||
        (rc = upload(P.d_fft, P.fft.data(), sizeof(PwFft) * P.fft.size())) ||
        (rc = upload(P.d_fftof, P.fft_of.data(), 4 * P.fft_of.size())) ||
        (rc = upload(P.d_tw, tw.data(), 16 * tw.size())) || (rc = upload(P.d_perm, perm.data(), 4 * perm.size())) ||
        (rc = upload(P.d_gpre, gpre.data(), 8 * gpre.size())))
        return rc;
    return IFS_OK;
}

int pw_build(ifs_ctx *c, PwLevel &P, int isg) {
    const int L = P.L;
    // every degree up to 4 L
    int rc = pw_grid(c, P, L + 1, 2 * L + 0.5, 2 * L, L);
    if (rc) return rc;
    // offsets -> canonical table: turned and mirrored about z until x >= y >= 0, and z >= 0
    std::map<std::array<int, 3>, int> canon;
    P.map.assign(216, PwMaps{});
    std::vector<char> used(216 * 8, 0);
    for (auto &S : P.src)
        for (int ch = 0; ch < 8; ++ch)
            if (S.mask >> ch & 1) used[S.r * 8 + ch] = 1;
    for (int r = 0; r < 216; ++r)
        for (int ch = 0; ch < 8; ++ch) {
            if (!used[r * 8 + ch]) continue;
            const int o[3] = {r / 36 - 2 - (ch >> 2), r / 6 % 6 - 2 - (ch >> 1 & 1), r % 6 - 2 - (ch & 1)};
            // direction of the phase factor: the translation vector isg * o turned by pi about z
            int v[3] = {-isg * o[0], -isg * o[1], isg * o[2]};
            PwMap M{0, v[2] < 0, 1, 0};
            int a = v[0], b = v[1], q = 0;
            while (!(a > 0 && b >= 0) && !(a == 0 && b == 0)) {  // turn by -pi/2 into the first quadrant
                const int t = a;
                a = b;
                b = -t;
                ++q;
            }
            // (a, b) = turn by -q quarters of v; mirror about the diagonal: angle -> pi/2 - angle
            // (i -> i - q N / 4, mirrored: -(i - (q + 1) N / 4))
            M.shift = -q;
            if (b > a) {
                std::swap(a, b);
                M.shift = (q + 1) & 3;
                M.sign = -1;
            }
            const std::array<int, 3> key = {a, b, std::abs(v[2])};
            auto it = canon.find(key);
            if (it == canon.end()) {
                it = canon.emplace(key, (int)P.canon.size()).first;
                P.canon.push_back(key);
            }
            M.table = it->second;
            P.map[r].child[ch] = M;
        }
    const int nc = (int)P.canon.size();
    std::vector<double> dir(4 * nc), t(nc);
    std::vector<int32_t> terms(nc);
    for (int i = 0; i < nc; ++i) {
        const auto &q = P.canon[i];
        const double r = std::sqrt((double)(q[0] * q[0] + q[1] * q[1] + q[2] * q[2]));
        for (int d = 0; d < 3; ++d) dir[4 * i + d] = q[d] / r;
        t[i] = P.k * (P.edge * r);
        terms[i] = pw_terms(P.k, P.edge, q[0] * q[0] + q[1] * q[1] + q[2] * q[2], L);
    }
    if ((rc = upload(P.d_src, P.src.data(), sizeof(PwSource) * P.src.size())) ||
        (rc = upload(P.d_par, P.par.data(), sizeof(PwParent) * P.par.size())) ||
        (rc = upload(P.d_map, P.map.data(), sizeof(PwMaps) * P.map.size())) ||
        (rc = upload(P.d_canon, dir.data(), 8 * dir.size())))
        return rc;
    // c_p of every table; t and the last terms lie behind them
    if ((rc = P.d_hank.alloc(16 * (size_t)nc * (2 * L + 1) + 12 * (size_t)nc))) return rc;
    double *dt = (double *)(P.d_hank.as<double2>() + (size_t)nc * (2 * L + 1));
    if (hipMemcpy(dt, t.data(), 8 * (size_t)nc, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dt + nc, terms.data(), 4 * (size_t)nc, hipMemcpyHostToDevice) != hipSuccess)
        return IFS_E_HIP;
    launch_pw_hankel(nc, 2 * L, dt, (const int32_t *)(dt + nc), P.d_hank.as<double2>(), c->stream);
    const size_t ub = 8 * (size_t)pw_ucnt(L + 1, L) * 2 * P.Q2, tb = 16 * (size_t)nc * P.SN;
    P.kept = ub + tb + c->ws_cached <= c->cache_budget;
    if (P.kept) {
        if (P.own_U.alloc(ub) || P.own_T.alloc(tb)) {
            for (DevBuf *d : {&P.own_U, &P.own_T})
                if (d->p) {
                    (void)hipFree(d->p);
                    d->p = nullptr;
                    d->bytes = 0;
                }
            P.kept = false;
        } else {
            c->ws_cached += ub + tb;
        }
    }
    if (hipPeekAtLastError() != hipSuccess) return IFS_E_HIP;
    return pw_prepare(c, P, 1, c->prm.precision);
}

int pw_plan(ifs_ctx *c, PwLevel &P, int nrhs) {
    P.plan_nrhs = 0;
    const int L = P.L, nc = (int)P.canon.size();
    const int64_t nbr = (int64_t)P.nb * nrhs;
    P.n_x = x_size(L) * nbr;
    const double left = (double)c->ws_budget - 32.0 * (double)P.n_x;
    P.chunks.clear();
    std::vector<int64_t> cpre;
    P.cpre_at.clear();
    P.n_g = P.n_f = P.n_u = P.n_t = 0;
    for (int j = 0; j < P.Q2;) {
        PwLevel::Chunk ch{j, 0, 0, 0, 0.0, 0.0};
        double bytes = 0.0;
        while (j + ch.R2 < P.Q2) {
            const int n = P.N[j + ch.R2];
            double b = 16.0 * 4.0 * (2 * L + 1) * (double)nbr + 16.0 * 8.0 * n * (double)nbr;
            if (!P.kept) b += 16.0 * (double)pw_ucnt(L + 1, L) + 32.0 * n * nc;
            if (ch.R2 > 0 && bytes + b > left) break;
            bytes += b;
            ch.sn += 2 * n;
            ch.maxN = std::max(ch.maxN, n);
            double gemm, fft;
            pw_row_flops(L, P.mF[j + ch.R2], n, gemm, fft);
            ch.f_gemm += gemm;
            ch.f_fft += fft;
            ++ch.R2;
        }
        P.cpre_at.push_back((int64_t)cpre.size());
        int64_t pre = 0;
        for (int lr = 0; lr < 2 * ch.R2; ++lr) {
            cpre.push_back(pre);
            pre += P.N[j + lr % ch.R2];
        }
        P.n_g = std::max(P.n_g, (int64_t)(2 * L + 1) * 4 * ch.R2 * nbr);
        P.n_f = std::max(P.n_f, 2 * ch.sn * nbr);
        P.n_u = std::max(P.n_u, pw_ucnt(L + 1, L) * 2 * ch.R2);
        P.n_t = std::max(P.n_t, ch.sn * nc);
        P.chunks.push_back(ch);
        j += ch.R2;
    }
    int rc;
    P.ws.y = 16 * (size_t)(2 * P.n_x + P.n_g);
    P.ws.z = 32 * (size_t)P.n_f;
    P.ws.d = P.kept ? 0 : 8 * (size_t)P.n_u;
    P.ws.ax = P.kept ? 0 : 16 * (size_t)P.n_t;
    if ((rc = ws_reserve(c, P.ws))) return rc;
    if ((rc = upload(P.d_cpre, cpre.data(), 8 * cpre.size()))) return rc;
    P.plan_nrhs = nrhs;
    return IFS_OK;
}

PwArg pw_arg(ifs_ctx *c, const PwLevel &P, int nrhs) {
    PwArg a{};
    a.L = P.L;
    a.nbr = P.nb * nrhs;
    a.Q2 = P.Q2;
    a.jlo = P.d_jlo.as<int32_t>();
    a.mF = P.d_mF.as<int32_t>();
    a.N = P.d_N.as<int32_t>();
    a.fftof = P.d_fftof.as<int32_t>();
    a.fft = P.d_fft.as<PwFft>();
    a.tw = P.d_tw.as<double2>();
    a.perm = P.d_perm.as<int32_t>();
    a.X = c->ws_y.as<double2>();
    a.Xd = a.X + P.n_x;
    a.G = a.Xd + P.n_x;
    a.F = c->ws_z.as<double2>();
    a.H = a.F + P.n_f;
    return a;
}

int pw_prepare(ifs_ctx *c, PwLevel &P, int nrhs, int prec) {
    if (prec == 1 && P.kept && !P.own_T32.p && !P.no_t32) {
        if (!capturing(c)) {
            const size_t b = 8 * P.canon.size() * (size_t)P.SN;
            P.no_t32 = b + c->ws_cached > c->cache_budget || P.own_T32.alloc(b) != IFS_OK;
            if (!P.no_t32) c->ws_cached += b;
        }
    }
    const int g = pw_group(c, P, nrhs);
    if (P.plan_nrhs != g) {
        if (hipStreamSynchronize(c->stream) != hipSuccess) return IFS_E_HIP;
        int rc = pw_plan(c, P, g);
        if (rc) return rc;
    }
    return ws_reserve(c, P.ws);
}

int pw_run(ifs_ctx *c, PwLevel &P, const double2 *C, double2 *D, int nrhs, int64_t stride, int prec) {
    const int g = pw_group(c, P, nrhs);
    if (int rc = pw_prepare(c, P, nrhs, prec)) return rc;
    for (int r0 = 0; r0 < nrhs; r0 += g) {
        const int nr = std::min(g, nrhs - r0);
        hipStream_t s = c->stream;
        const int L = P.L, nc = (int)P.canon.size();
        PwArg a = pw_arg(c, P, nr);
        const double *mu = P.d_mu.as<double>();
        double *U = P.kept ? P.own_U.as<double>() : c->ws_d.as<double>();
        double2 *T = P.kept ? P.own_T.as<double2>() : c->ws_ax.as<double2>();
        a.U = U;
        a.T = T;
        float2 *T32 = prec != 1 ? nullptr : P.kept ? P.own_T32.as<float2>() : (float2 *)T;
        a.T32 = T32;
        auto tables = [&](int j0, int R2, int maxN, bool u, bool t) {
            Scope sc(c, "m2l_gen_tables");
            if (u) launch_pw_utable(L, P.Q2, j0, R2, a.a0, a.a1, a.ustr, mu, U, s);
            if (t)
                launch_pw_ttable(nc, 2 * L, P.Q2, j0, R2, a.a0, a.a1, maxN, mu, P.d_canon.as<double>(), a.N, a.tpre,
                                 a.tsn, P.d_hank.as<double2>(), T, T32, s);
        };
        if (P.kept) {
            a.tpre = P.d_gpre.as<int64_t>();
            a.tsn = P.SN;
            a.ustr = 2 * P.Q2;
            const int t = T32 ? 1 : 0;
            if (!P.ready || !P.t_ready[t]) {
                a.a0 = 0;
                a.a1 = P.Q2;
                tables(0, P.Q2, *std::max_element(P.N.begin(), P.N.end()), !P.ready, !P.t_ready[t]);
                if (!capturing(c)) P.ready = P.t_ready[t] = true;
            }
        }
        {
            Scope sc(c, "m2l_pack");
            launch_pw_pack(a, P.nb, P.off, C + r0 * stride, stride, s);
        }
        for (size_t i = 0; i < P.chunks.size(); ++i) {
            const auto &ch = P.chunks[i];
            a.j0 = ch.j0;
            a.R2 = ch.R2;
            a.cpre = P.d_cpre.as<int64_t>() + P.cpre_at[i];
            if (P.kept) {
                a.a0 = ch.j0;
                a.a1 = P.Q2 + ch.j0;
            } else {
                a.a0 = 0;
                a.a1 = ch.R2;
                a.ustr = 2 * ch.R2;
                a.tpre = a.cpre;
                a.tsn = ch.sn;
                tables(ch.j0, ch.R2, ch.maxN, true, true);
            }
            const double nbr = (double)P.nb * nr;
            {
                Scope sc(c, "m2l_synth", ch.f_gemm * nbr);
                launch_pw_synth(a, s);
            }
            {
                Scope sc(c, "m2l_fft", ch.f_fft * nbr);
                launch_pw_fft(a, 0, ch.maxN, s);
            }
            {
                Scope sc(c, "m2l_product", 16.0 * (double)ch.sn * (double)P.ncols * nr);
                launch_pw_m2l(a, P.d_par.as<PwParent>(), (int)P.par.size(), P.d_src.as<PwSource>(), P.d_map.as<PwMaps>(),
                              P.nb, nr, ch.maxN, s);
            }
            {
                Scope sc(c, "m2l_fft", ch.f_fft * nbr);
                launch_pw_fft(a, 1, ch.maxN, s);
            }
            {
                Scope sc(c, "m2l_anal", ch.f_gemm * nbr);
                launch_pw_anal(a, i > 0, s);
            }
        }
        {
            Scope sc(c, "m2l_unpack");
            launch_pw_unpack(a, P.nb, P.off, D + r0 * stride, stride, s);
        }
    }
    return hipPeekAtLastError() == hipSuccess ? IFS_OK : IFS_E_HIP;
}

void pw_row_flops(int L, int mF, int N, double &gemm, double &fft) {
    gemm = 16.0 * (double)(pw_xcnt(mF, L) + pw_cn(mF, L) - pw_xcnt(-mF, L));
    fft = 20.0 * N * std::log2((double)N);
}

double pw_flops(const PwLevel &P) {
    double box = 0.0;
    for (int j = 0; j < P.Q2; ++j) {
        double gemm, fft;
        pw_row_flops(P.L, P.mF[j], P.N[j], gemm, fft);
        box += 2.0 * (gemm + fft);
    }
    return box * P.nb + 16.0 * (double)P.SN * (double)P.ncols;
}

uint64_t pw_sig(const PwLevel &P) {
    uint64_t h = (uint64_t)P.plan_nrhs;
    for (const DevBuf *d : {&P.d_mu, &P.d_src, &P.d_par, &P.d_cpre, &P.d_hank, &P.own_U, &P.own_T, &P.own_T32})
        h ^= (uint64_t)(uintptr_t)d->p + 0x9e3779b97f4a7c15ull + (h << 6) + (h >> 2);
    return h;
}

}  // namespace ifs
