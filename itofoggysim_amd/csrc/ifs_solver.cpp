// Restarted GMRES on the device (FP64), the plane-wave right-hand side, and the
// remaining C ABI entry points.
//
// The reference drives CERFACS ZGMRES by reverse communication with modified
// Gram-Schmidt and zgemv dot products (FoggySim/src/lib/mie_theory/lib_solver_GMRES.f90:116-316).
// Here the Krylov basis lives in HBM; orthogonalisation is classical Gram-Schmidt
// with one re-orthogonalisation pass (batched dot products, fixed reduction
// order), and the small Hessenberg / Givens update runs on the host in FP64.
//
// The iteration runs in the normalised basis x_hat = S x, s(n,m) =
// sqrt(n(n+1)(2n+1)(n-m)!/(n+m)!), where the operator is S (I + T A) S^-1.  In
// Xu's basis the entries of A span ~1e+-96 at n ~ 20 (factorial ratios), and
// Krylov iterations under the plain 2-norm stall; the tolerance therefore refers
// to the relative residual in the normalised basis.
#include <hip/hip_runtime.h>

#include <chrono>
#include <cstdio>
#include <cmath>
#include <complex>
#include <vector>

#include "../../include/ifs.h"
#include "ifs_engine.h"
#include "ifs_internal.h"

using namespace ifs;
using cplx = std::complex<double>;

// Accessors implemented in ifs_api.cpp
namespace ifs {
hipStream_t ctx_stream(ifs_ctx *c);
int ctx_krylov_alloc(ifs_ctx *c, int restart, int64_t n, double2 **V, double2 **w, double2 **r, double2 **part,
                     double2 **h);
double2 *c_bhat(ifs_ctx *c, int64_t n);
double2 *c_xhat(ifs_ctx *c, int64_t n);
double2 *c_stage(ifs_ctx *c, int64_t n);
int ctx_ns(ifs_ctx *c);
int ctx_N(ifs_ctx *c);
const double *ctx_pos(ifs_ctx *c);
double ctx_k(ifs_ctx *c);
int scale_flat(ifs_ctx *c, const double2 *x, double2 *y, int inverse);
double flat_rel_residual(ifs_ctx *c, const double2 *r_hat, const double2 *b_hat, int64_t n);
}  // namespace ifs

namespace {

int fetch(hipStream_t s, const double2 *d, int cnt, cplx *out) {
    if (hipMemcpyAsync(out, d, sizeof(double2) * cnt, hipMemcpyDeviceToHost, s) != hipSuccess) return IFS_E_HIP;
    return hipStreamSynchronize(s) == hipSuccess ? IFS_OK : IFS_E_HIP;
}

int dots(hipStream_t s, const double2 *V, int64_t ldv, int nv, const double2 *w, int64_t n, double2 *d_out,
         double2 *d_part, std::vector<cplx> &out) {
    launch_dots(V, ldv, nv, w, n, d_out, d_part, s);
    out.resize(nv);
    return fetch(s, d_out, nv, out.data());
}

// Classical Gram-Schmidt with one re-orthogonalisation pass, enqueued as a whole: the
// coefficients of both passes and |w|^2 of the result stay on the device (h: 2 nv + 1
// entries) and are read once, by cgs2_fetch.
void cgs2(hipStream_t s, const double2 *V, int64_t ldv, int nv, double2 *w, int64_t n, double2 *h, double2 *d_part) {
    launch_dots(V, ldv, nv, w, n, h, d_part, s);
    launch_gemv_sub(V, ldv, nv, h, w, n, nullptr, nullptr, s);
    launch_dots(V, ldv, nv, w, n, h + nv, d_part, s);
    launch_gemv_sub(V, ldv, nv, h + nv, w, n, h + 2 * nv, d_part, s);
}

// coefficients (sum of both passes) into hv, |w| returned; h on the host
double cgs2_sum(const cplx *h, int nv, std::vector<cplx> &hv) {
    hv.resize(nv);
    for (int i = 0; i < nv; ++i) hv[i] = h[i] + h[nv + i];
    return std::sqrt(std::max(0.0, h[2 * nv].real()));
}

double norm2(hipStream_t s, const double2 *w, int64_t n, double2 *d_out, double2 *d_part, int &rc) {
    std::vector<cplx> o;
    rc = dots(s, w, n, 1, w, n, d_out, d_part, o);
    return std::sqrt(std::max(0.0, o[0].real()));
}

}  // namespace

extern "C" int ifs_solve_device(ifs_ctx *c, const void *rhs_dev, void *x_dev, int64_t n, const ifs_solve_opts *opts,
                                ifs_solve_info *info) {
    if (!c || !rhs_dev || !x_dev || !opts || n != ifs_vector_length(c)) return IFS_E_ARG;
    const int m = opts->restart;
    if (m < 1 || opts->max_iter < 1 || !(opts->tol > 0.0)) return IFS_E_ARG;
    if (opts->precision != IFS_PREC_FP64 && opts->precision != IFS_PREC_MIXED) return IFS_E_ARG;
    // Arnoldi products in the requested precision; the true residual of every cycle in FP64
    const int kprec = opts->precision == IFS_PREC_MIXED ? 1 : 0;
    auto t0 = std::chrono::steady_clock::now();
    hipStream_t s = ctx_stream(c);
    double2 *V, *w, *r, *part, *h;
    int rc = ctx_krylov_alloc(c, m, n, &V, &w, &r, &part, &h);
    if (rc) return rc;
    const double2 *b_in = (const double2 *)rhs_dev;
    double2 *x_out = (double2 *)x_dev;
    // normalised right-hand side and iterate live in the Krylov workspace
    double2 *b = c_bhat(c, n), *x = c_xhat(c, n);
    if (!b || !x) return IFS_E_NOMEM;
    if ((rc = scale_flat(c, b_in, b, 0))) return rc;
    if (opts->use_x0 && (rc = scale_flat(c, x_out, x, 0))) return rc;
    const double2 one = make_double2(1.0, 0.0), mone = make_double2(-1.0, 0.0), zero = make_double2(0.0, 0.0);

    double bnorm = norm2(s, b, n, h, part, rc);
    if (rc) return rc;
    int iters = 0;
    if (!opts->use_x0) launch_zero(x, n, s);
    if (bnorm == 0.0) {
        launch_zero(x_out, n, s);
        if (info) *info = {0, 1, 0.0, 0.0, 0.0};
        return IFS_OK;
    }
    // graph mode: the Arnoldi products go through one staging vector, so that one
    // captured matvec serves every Krylov vector
    const bool graph = (opts->flags & IFS_SOLVE_GRAPH) != 0;
    double2 *stage = graph ? c_stage(c, n) : nullptr;  // context-owned: later solves replay the same graph
    if (graph && !stage) return IFS_E_NOMEM;
    // r = b - M x
    auto residual = [&]() -> int {
        int q = graph ? matvec_graph(c, x, r, 1, 1, n) : matvec_impl(c, x, r, 1, 1, n);
        if (q) return q;
        ++iters;
        launch_axpby(one, b, mone, r, n, s);
        return IFS_OK;
    };
    // with x = 0 the first residual is b itself (no product)
    if (opts->use_x0) {
        if ((rc = residual())) return rc;
    } else {
        launch_scale_copy(one, b, r, n, s);
    }
    double beta = norm2(s, r, n, h, part, rc);
    if (rc) return rc;
    std::vector<cplx> H((size_t)(m + 1) * m), g(m + 1), cs(m), sn(m), hv, hh(2 * m + 1);
    int converged = beta / bnorm < opts->tol;
    int breakdown = 0;
    while (!converged && iters < opts->max_iter) {
        launch_scale_copy(make_double2(1.0 / beta, 0.0), r, V, n, s);
        std::fill(g.begin(), g.end(), cplx(0.0));
        g[0] = beta;
        int jend = 0;
        for (int j = 0; j < m; ++j) {
            double2 *vj = V + (int64_t)j * n;
            if (graph) {
                launch_scale_copy(one, vj, stage, n, s);
                rc = matvec_graph(c, stage, w, 1, 1, n, -1, kprec);
            } else {
                rc = matvec_impl(c, vj, w, 1, 1, n, -1, kprec);
            }
            if (rc) return rc;
            ++iters;
            cgs2(s, V, n, j + 1, w, n, h, part);
            if ((rc = fetch(s, h, 2 * j + 3, hh.data()))) return rc;
            const double hn = cgs2_sum(hh.data(), j + 1, hv);
            // Hessenberg column j, previous rotations, new rotation
            for (int i = 0; i <= j; ++i) H[(size_t)i * m + j] = hv[i];
            H[(size_t)(j + 1) * m + j] = hn;
            for (int i = 0; i < j; ++i) {
                cplx a = H[(size_t)i * m + j], bb = H[(size_t)(i + 1) * m + j];
                H[(size_t)i * m + j] = cs[i] * a + sn[i] * bb;
                H[(size_t)(i + 1) * m + j] = -std::conj(sn[i]) * a + cs[i] * bb;
            }
            cplx a = H[(size_t)j * m + j], bb = H[(size_t)(j + 1) * m + j];
            double ra = std::abs(a), rb = std::abs(bb), rr = std::hypot(ra, rb);
            if (rr == 0.0) {
                cs[j] = 1.0;
                sn[j] = 0.0;
            } else if (ra == 0.0) {
                cs[j] = 0.0;
                sn[j] = std::conj(bb) / rb;
                H[(size_t)j * m + j] = rb;
            } else {
                cs[j] = ra / rr;
                sn[j] = (a / ra) * std::conj(bb) / rr;
                H[(size_t)j * m + j] = (a / ra) * rr;
            }
            H[(size_t)(j + 1) * m + j] = 0.0;
            g[j + 1] = -std::conj(sn[j]) * g[j];
            g[j] = cs[j] * g[j];
            jend = j + 1;
            double est = std::abs(g[j + 1]) / bnorm;
            if (opts->verbose && iters % 5 == 0) {
                double el = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
                std::fprintf(stderr, "gmres: %d matvecs, estimated rel residual %.3e, %.1f s\n", iters, est, el);
                std::fflush(stderr);
            }
            if (hn == 0.0) {
                breakdown = 1;
                break;
            }
            if (est < opts->tol || iters >= opts->max_iter) break;
            launch_scale_copy(make_double2(1.0 / hn, 0.0), w, V + (int64_t)(j + 1) * n, n, s);
        }
        // y = H^-1 g (upper triangular), x += V y
        std::vector<cplx> y(jend);
        for (int i = jend - 1; i >= 0; --i) {
            cplx acc = g[i];
            for (int k = i + 1; k < jend; ++k) acc -= H[(size_t)i * m + k] * y[k];
            y[i] = acc / H[(size_t)i * m + i];
        }
        if (hipMemcpyAsync(h, y.data(), sizeof(double2) * jend, hipMemcpyHostToDevice, s) != hipSuccess)
            return IFS_E_HIP;
        launch_gemv_add(V, n, jend, h, x, n, s);
        // true residual in FP64
        if ((rc = residual())) return rc;
        beta = norm2(s, r, n, h, part, rc);
        if (rc) return rc;
        converged = beta / bnorm < opts->tol;
        if (opts->verbose) {
            double el = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
            std::fprintf(stderr, "gmres: %d matvecs, true rel residual %.3e, %.1f s\n", iters, beta / bnorm, el);
            std::fflush(stderr);
        }
        if (breakdown && !converged) break;
        (void)zero;
    }
    if ((rc = scale_flat(c, x, x_out, 1))) return rc;
    if (hipStreamSynchronize(s) != hipSuccess) return IFS_E_HIP;
    double secs = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    if (info) {
        info->iterations = iters;
        info->converged = converged;
        info->rel_residual = beta / bnorm;
        info->seconds = secs;
        // r holds the last true residual b_hat - M_hat x_hat
        info->rel_residual_flat = flat_rel_residual(c, r, b, n);
    }
    if (converged) return IFS_OK;
    return breakdown ? IFS_E_BREAKDOWN : IFS_E_NOCONV;
}

namespace {

// Independent linear systems advanced in lock step.  The vectors the operator acts on
// are `ncols` columns of length `ncol`; system r is the entries [off[r], off[r] +
// len[r]) of column col[r].  Many right-hand sides of one cluster: one system per
// column, each the whole column.  Independent clusters in one context (a block-
// diagonal operator): one column, one system per cluster's entries.
struct Systems {
    int ncols = 1;
    int64_t ncol = 0;
    std::vector<int> col;
    std::vector<int64_t> off, len;
    int size() const { return (int)col.size(); }
};

// Restarted GMRES for every system in lock step: each Arnoldi step applies the
// operator to the current Krylov vectors of all systems in one matvec call (one
// batched product over the columns; the translation tables serve every column and
// every cluster); orthogonalisation (CGS2), Givens rotations and the true-residual
// test stay per system.  A system that converged keeps riding along in the products
// until all are done, and its iterate no longer changes.
int solve_systems(ifs_ctx *c, const Systems &L, const double2 *bin, double2 *xout, int64_t ld,
                  const ifs_solve_opts *opts, ifs_solve_info *info) {
    const int m = opts->restart;
    const int kprec = opts->precision == IFS_PREC_MIXED ? 1 : 0;
    const int ns = L.size(), nc = L.ncols;
    const int64_t n = L.ncol;
    auto t0 = std::chrono::steady_clock::now();
    hipStream_t s = ctx_stream(c);
    DevBuf dV, dW, dR, dB, dX, dpart, dh;
    int rc;
    const int64_t ldv = (int64_t)(m + 1) * n;  // V[column][j][n]
    if ((rc = dV.alloc(16ull * ldv * nc)) || (rc = dW.alloc(16ull * n * nc)) || (rc = dR.alloc(16ull * n * nc)) ||
        (rc = dB.alloc(16ull * n * nc)) || (rc = dX.alloc(16ull * n * nc)) ||
        (rc = dpart.alloc(16ull * kDotMax * (m + 1))) || (rc = dh.alloc(16ull * (2 * m + 1) * ns)))
        return rc;
    double2 *V = dV.as<double2>(), *W = dW.as<double2>(), *R = dR.as<double2>(), *B = dB.as<double2>(),
            *X = dX.as<double2>(), *part = dpart.as<double2>(), *h = dh.as<double2>();
    launch_zero(V, ldv * nc, s);
    const bool graph = (opts->flags & IFS_SOLVE_GRAPH) != 0;
    DevBuf dstage;
    if (graph && (rc = dstage.alloc(16ull * n * nc))) return rc;
    double2 *stage = dstage.as<double2>();
    // system r's entries in a column vector, and its Krylov vector j
    auto at = [&](double2 *base, int r) { return base + (int64_t)L.col[r] * n + L.off[r]; };
    auto kv = [&](int r, int j) { return V + (int64_t)L.col[r] * ldv + (int64_t)j * n + L.off[r]; };
    const double2 one = make_double2(1.0, 0.0), mone = make_double2(-1.0, 0.0);
    std::vector<double> bnorm(ns), beta(ns), flat(ns, 0.0);
    std::vector<int> iters(ns, 0), conv(ns, 0), brk(ns, 0);
    for (int q = 0; q < nc; ++q) {
        if ((rc = scale_flat(c, bin + q * ld, B + q * n, 0))) return rc;
        if (opts->use_x0) {
            if ((rc = scale_flat(c, xout + q * ld, X + q * n, 0))) return rc;
        } else {
            launch_zero(X + q * n, n, s);
        }
    }
    for (int r = 0; r < ns; ++r) {
        bnorm[r] = norm2(s, at(B, r), L.len[r], h, part, rc);
        if (rc) return rc;
    }
    // first: with x = 0 the residual is b itself (no product)
    auto residual = [&](bool first) -> int {
        int q = IFS_OK;
        if (!first || opts->use_x0) {
            q = graph ? matvec_graph(c, X, R, 1, nc, n) : matvec_impl(c, X, R, 1, nc, n);
            if (q) return q;
        }
        for (int r = 0; r < ns; ++r) {
            if (conv[r]) continue;
            if (!first || opts->use_x0) {
                ++iters[r];
                launch_axpby(one, at(B, r), mone, at(R, r), L.len[r], s);
            } else {
                launch_scale_copy(one, at(B, r), at(R, r), L.len[r], s);
            }
            beta[r] = norm2(s, at(R, r), L.len[r], h, part, q);
            if (q) return q;
            conv[r] = bnorm[r] == 0.0 || beta[r] / bnorm[r] < opts->tol;
            // the flat-basis residual of this true residual (R of a converged system is
            // overwritten by later products)
            flat[r] = bnorm[r] > 0.0 ? flat_rel_residual(c, at(R, r), at(B, r), L.len[r]) : 0.0;
        }
        return IFS_OK;
    };
    if ((rc = residual(true))) return rc;
    struct St {
        std::vector<cplx> H, g, cs, sn;
        int jend = 0;
        bool done = false;
    };
    std::vector<St> st(ns);
    auto active = [&](int r) { return !conv[r] && !brk[r] && iters[r] < opts->max_iter; };
    std::vector<cplx> hv, hh((size_t)(2 * m + 1) * ns);
    for (;;) {
        bool any = false;
        for (int r = 0; r < ns; ++r) any = any || active(r);
        if (!any) break;
        for (int r = 0; r < ns; ++r) {
            St &S = st[r];
            S.done = !active(r);
            S.jend = 0;
            if (S.done) continue;
            S.H.assign((size_t)(m + 1) * m, 0.0);
            S.g.assign(m + 1, 0.0);
            S.cs.assign(m, 0.0);
            S.sn.assign(m, 0.0);
            S.g[0] = beta[r];
            launch_scale_copy(make_double2(1.0 / beta[r], 0.0), at(R, r), kv(r, 0), L.len[r], s);
        }
        for (int j = 0; j < m; ++j) {
            bool work = false;
            for (int r = 0; r < ns; ++r) work = work || !st[r].done;
            if (!work) break;
            // w = M v_j for every column in one call
            if (graph) {
                for (int q = 0; q < nc; ++q) launch_scale_copy(one, V + q * ldv + (int64_t)j * n, stage + q * n, n, s);
                rc = matvec_graph(c, stage, W, 1, nc, n, n, kprec);
            } else {
                rc = matvec_impl(c, V + (int64_t)j * n, W, 1, nc, ldv, n, kprec);
            }
            if (rc) return rc;
            // every system's orthogonalisation is enqueued before the one read of all coefficients
            const int hs = 2 * j + 3;
            for (int r = 0; r < ns; ++r)
                if (!st[r].done) cgs2(s, kv(r, 0), n, j + 1, at(W, r), L.len[r], h + (int64_t)r * hs, part);
            if ((rc = fetch(s, h, ns * hs, hh.data()))) return rc;
            for (int r = 0; r < ns; ++r) {
                St &S = st[r];
                if (S.done) continue;
                ++iters[r];
                double2 *w = at(W, r);
                const int64_t len = L.len[r];
                const double hn = cgs2_sum(hh.data() + (size_t)r * hs, j + 1, hv);
                std::vector<cplx> &H = S.H;
                for (int i = 0; i <= j; ++i) H[(size_t)i * m + j] = hv[i];
                H[(size_t)(j + 1) * m + j] = hn;
                for (int i = 0; i < j; ++i) {
                    cplx a = H[(size_t)i * m + j], bb = H[(size_t)(i + 1) * m + j];
                    H[(size_t)i * m + j] = S.cs[i] * a + S.sn[i] * bb;
                    H[(size_t)(i + 1) * m + j] = -std::conj(S.sn[i]) * a + S.cs[i] * bb;
                }
                cplx a = H[(size_t)j * m + j], bb = H[(size_t)(j + 1) * m + j];
                double ra = std::abs(a), rb = std::abs(bb), rr = std::hypot(ra, rb);
                if (rr == 0.0) {
                    S.cs[j] = 1.0;
                    S.sn[j] = 0.0;
                } else if (ra == 0.0) {
                    S.cs[j] = 0.0;
                    S.sn[j] = std::conj(bb) / rb;
                    H[(size_t)j * m + j] = rb;
                } else {
                    S.cs[j] = ra / rr;
                    S.sn[j] = (a / ra) * std::conj(bb) / rr;
                    H[(size_t)j * m + j] = (a / ra) * rr;
                }
                H[(size_t)(j + 1) * m + j] = 0.0;
                S.g[j + 1] = -std::conj(S.sn[j]) * S.g[j];
                S.g[j] = S.cs[j] * S.g[j];
                S.jend = j + 1;
                double est = std::abs(S.g[j + 1]) / bnorm[r];
                if (hn == 0.0) {
                    brk[r] = 1;
                    S.done = true;
                } else if (est < opts->tol || iters[r] >= opts->max_iter || j + 1 == m) {
                    S.done = true;
                } else {
                    launch_scale_copy(make_double2(1.0 / hn, 0.0), w, kv(r, j + 1), len, s);
                }
            }
            if (opts->verbose) {
                int nact = 0;
                for (int r = 0; r < ns; ++r) nact += !st[r].done;
                double el = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
                std::fprintf(stderr, "gmres: %d systems, step %d, %d still in the cycle, %.1f s\n", ns, j + 1, nact,
                             el);
                std::fflush(stderr);
            }
        }
        for (int r = 0; r < ns; ++r) {
            St &S = st[r];
            if (S.jend == 0) continue;
            std::vector<cplx> y(S.jend);
            for (int i = S.jend - 1; i >= 0; --i) {
                cplx acc = S.g[i];
                for (int k = i + 1; k < S.jend; ++k) acc -= S.H[(size_t)i * m + k] * y[k];
                y[i] = acc / S.H[(size_t)i * m + i];
            }
            if (hipMemcpyAsync(h, y.data(), sizeof(double2) * S.jend, hipMemcpyHostToDevice, s) != hipSuccess)
                return IFS_E_HIP;
            launch_gemv_add(kv(r, 0), n, S.jend, h, at(X, r), L.len[r], s);
        }
        if ((rc = residual(false))) return rc;
        for (int r = 0; r < ns; ++r)
            if (brk[r] && conv[r]) brk[r] = 0;
    }
    for (int q = 0; q < nc; ++q)
        if ((rc = scale_flat(c, X + q * n, xout + q * ld, 1))) return rc;
    if (hipStreamSynchronize(s) != hipSuccess) return IFS_E_HIP;
    double secs = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    int all = 1, anybrk = 0;
    for (int r = 0; r < ns; ++r) {
        if (info) {
            info[r].iterations = iters[r];
            info[r].converged = conv[r];
            info[r].rel_residual = bnorm[r] > 0.0 ? beta[r] / bnorm[r] : 0.0;
            info[r].seconds = secs;
            info[r].rel_residual_flat = flat[r];
        }
        all = all && conv[r];
        anybrk = anybrk || brk[r];
    }
    if (all) return IFS_OK;
    return anybrk ? IFS_E_BREAKDOWN : IFS_E_NOCONV;
}

int check_opts(const ifs_solve_opts *opts) {
    if (opts->restart < 1 || opts->max_iter < 1 || !(opts->tol > 0.0)) return IFS_E_ARG;
    if (opts->precision != IFS_PREC_FP64 && opts->precision != IFS_PREC_MIXED) return IFS_E_ARG;
    return IFS_OK;
}

}  // namespace

// Block GMRES (restarted): the nrhs right-hand sides share one Krylov space,
//   K_m(M, R0) = span{R0, M R0, ..., M^{m-1} R0},  R0 = B - M X0  (n x p blocks),
// so every block step applies one batched product to p Krylov vectors and every right-
// hand side's iterate is corrected from all m p basis vectors.  Block Arnoldi with
// classical Gram-Schmidt against the basis (two passes) and modified Gram-Schmidt with
// re-orthogonalisation inside the new block gives the block Hessenberg matrix H (upper
// triangular p x p sub-diagonal blocks); Givens rotations reduce it column by column
// and minimise ||E1 S - H Y||_F for all right-hand sides together, whose column norms
// of the rotated residual block are the per-right-hand-side residual estimates.
// A direction that becomes dependent on the basis (norm below 1e-14 of the block's
// largest) is dropped: its basis vector is zero and contributes nothing.  The true
// residual of every restart cycle is recomputed with FP64 products.
static int solve_block(ifs_ctx *c, int p, const double2 *bin, double2 *xout, int64_t ld, const ifs_solve_opts *opts,
                       ifs_solve_info *info) {
    const int m = opts->restart;
    const int kprec = opts->precision == IFS_PREC_MIXED ? 1 : 0;
    const int64_t n = ifs_vector_length(c);
    const int mp = m * p, mp1 = (m + 1) * p;
    auto t0 = std::chrono::steady_clock::now();
    hipStream_t s = ctx_stream(c);
    DevBuf dV, dW, dR, dB, dX, dpart, dh;
    int rc;
    if ((rc = dV.alloc(16ull * n * mp1)) || (rc = dW.alloc(16ull * n * p)) || (rc = dR.alloc(16ull * n * p)) ||
        (rc = dB.alloc(16ull * n * p)) || (rc = dX.alloc(16ull * n * p)) ||
        (rc = dpart.alloc(16ull * kDotMax * mp1)) || (rc = dh.alloc(16ull * (2 * mp + 1))))
        return rc;
    double2 *V = dV.as<double2>(), *W = dW.as<double2>(), *R = dR.as<double2>(), *B = dB.as<double2>(),
            *X = dX.as<double2>(), *part = dpart.as<double2>(), *h = dh.as<double2>();
    const double2 one = make_double2(1.0, 0.0), mone = make_double2(-1.0, 0.0);
    std::vector<double> bnorm(p), beta(p), flat(p, 0.0);
    for (int q = 0; q < p; ++q) {
        if ((rc = scale_flat(c, bin + q * ld, B + q * n, 0))) return rc;
        if (opts->use_x0) {
            if ((rc = scale_flat(c, xout + q * ld, X + q * n, 0))) return rc;
        } else {
            launch_zero(X + q * n, n, s);
        }
        bnorm[q] = norm2(s, B + q * n, n, h, part, rc);
        if (rc) return rc;
    }
    std::vector<cplx> hh(2 * (size_t)mp);
    auto upload = [&](const std::vector<cplx> &v, int cnt) -> int {
        return hipMemcpyAsync(h, v.data(), sizeof(double2) * cnt, hipMemcpyHostToDevice, s) == hipSuccess ? IFS_OK
                                                                                                            : IFS_E_HIP;
    };
    // orthonormalises the p columns at Q (stride n) among themselves (MGS, two passes);
    // T[q' + p q] receives the upper-triangular factor (column-major p x p)
    auto block_qr = [&](double2 *Q, std::vector<cplx> &T) -> int {
        T.assign((size_t)p * p, 0.0);
        std::vector<double> nrm0(p);
        double big = 0.0;
        for (int q = 0; q < p; ++q) {
            int e = 0;
            nrm0[q] = norm2(s, Q + q * n, n, h, part, e);
            if (e) return e;
            big = std::max(big, nrm0[q]);
        }
        for (int q = 0; q < p; ++q) {
            double2 *w = Q + q * n;
            for (int pass = 0; pass < 2; ++pass)
                for (int r = 0; r < q; ++r) {
                    std::vector<cplx> d;
                    int e = dots(s, Q + r * n, n, 1, w, n, h, part, d);
                    if (e) return e;
                    T[r + (size_t)p * q] += d[0];
                    launch_axpby(make_double2(-d[0].real(), -d[0].imag()), Q + r * n, one, w, n, s);
                }
            int e = 0;
            double nr = norm2(s, w, n, h, part, e);
            if (e) return e;
            if (nr > 1e-14 * big && nr > 0.0) {
                T[q + (size_t)p * q] = nr;
                launch_scale_copy(make_double2(1.0 / nr, 0.0), w, w, n, s);
            } else {  // dependent direction: dropped
                T[q + (size_t)p * q] = 0.0;
                launch_zero(w, n, s);
            }
        }
        return IFS_OK;
    };
    int iters = 0;
    std::vector<int> conv(p, 0);
    bool first = true;
    for (;;) {
        // true residual R = B - M X in FP64
        if (!first || opts->use_x0) {
            if ((rc = matvec_impl(c, X, R, 1, p, n))) return rc;
            for (int q = 0; q < p; ++q) launch_axpby(one, B + q * n, mone, R + q * n, n, s);
            if (!first) ++iters;
        } else {
            for (int q = 0; q < p; ++q) launch_scale_copy(one, B + q * n, R + q * n, n, s);
        }
        first = false;
        bool all = true;
        for (int q = 0; q < p; ++q) {
            beta[q] = norm2(s, R + q * n, n, h, part, rc);
            if (rc) return rc;
            conv[q] = bnorm[q] == 0.0 || beta[q] / bnorm[q] < opts->tol;
            all = all && conv[q];
            flat[q] = bnorm[q] > 0.0 ? flat_rel_residual(c, R + q * n, B + q * n, n) : 0.0;
        }
        if (opts->verbose) {
            double worst = 0.0;
            for (int q = 0; q < p; ++q) worst = std::max(worst, bnorm[q] > 0.0 ? beta[q] / bnorm[q] : 0.0);
            double el = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
            std::fprintf(stderr, "block gmres: %d products, worst true rel residual %.3e, %.1f s\n", iters, worst, el);
            std::fflush(stderr);
        }
        if (all || iters >= opts->max_iter) break;
        // V_0 S = R
        if (hipMemcpyAsync(V, R, 16ull * n * p, hipMemcpyDeviceToDevice, s) != hipSuccess) return IFS_E_HIP;
        std::vector<cplx> S;
        if ((rc = block_qr(V, S))) return rc;
        // H: mp1 x mp (column-major), G: mp1 x p (column-major), Givens rotations in order
        std::vector<cplx> H((size_t)mp1 * mp, 0.0), G((size_t)mp1 * p, 0.0);
        for (int q = 0; q < p; ++q)
            for (int r = 0; r <= q; ++r) G[r + (size_t)mp1 * q] = S[r + (size_t)p * q];
        struct Rot {
            int k, i;
            double cs;
            cplx sn;
        };
        std::vector<Rot> rots;
        auto rot_apply = [&](const Rot &g, cplx &a, cplx &b) {
            const cplx x = a, y = b;
            a = g.cs * x + g.sn * y;
            b = -std::conj(g.sn) * x + g.cs * y;
        };
        int jend = 0;
        for (int j = 0; j < m; ++j) {
            // W = M V_j (p columns, one product)
            if ((rc = matvec_impl(c, V + (int64_t)j * p * n, W, 1, p, n, n, kprec))) return rc;
            ++iters;
            const int nb = (j + 1) * p;  // basis vectors so far
            for (int q = 0; q < p; ++q) {
                double2 *w = W + q * n;
                cplx *hc = &H[(size_t)mp1 * (j * p + q)];
                cgs2(s, V, n, nb, w, n, h, part);
                if ((rc = fetch(s, h, 2 * nb, hh.data()))) return rc;
                for (int i = 0; i < nb; ++i) hc[i] += hh[i] + hh[nb + i];
            }
            // V_{j+1} T = W
            std::vector<cplx> T;
            if ((rc = block_qr(W, T))) return rc;
            if (hipMemcpyAsync(V + (int64_t)nb * n, W, 16ull * n * p, hipMemcpyDeviceToDevice, s) != hipSuccess)
                return IFS_E_HIP;
            for (int q = 0; q < p; ++q)
                for (int r = 0; r <= q; ++r) H[(size_t)mp1 * (j * p + q) + nb + r] = T[r + (size_t)p * q];
            // reduce the new block column: every earlier rotation on all p new columns first,
            // then the new ones below the diagonal, each applied to the columns it reaches
            const size_t nold = rots.size();
            for (int q = 0; q < p; ++q) {
                cplx *hc = &H[(size_t)mp1 * (j * p + q)];
                for (size_t g = 0; g < nold; ++g) rot_apply(rots[g], hc[rots[g].k], hc[rots[g].i]);
            }
            for (int q = 0; q < p; ++q) {
                cplx *hc = &H[(size_t)mp1 * (j * p + q)];
                const int k = j * p + q;
                for (int i = k + 1; i <= nb + q; ++i) {
                    const cplx a = hc[k], b = hc[i];
                    const double ra = std::abs(a), rb = std::abs(b);
                    if (rb == 0.0) continue;
                    const double rr = std::hypot(ra, rb);
                    Rot g{k, i, 0.0, 0.0};
                    if (ra == 0.0) {
                        g.cs = 0.0;
                        g.sn = std::conj(b) / rb;
                    } else {
                        g.cs = ra / rr;
                        g.sn = (a / ra) * std::conj(b) / rr;
                    }
                    for (int q2 = q; q2 < p; ++q2) {
                        cplx *h2 = &H[(size_t)mp1 * (j * p + q2)];
                        rot_apply(g, h2[k], h2[i]);
                    }
                    hc[i] = 0.0;
                    for (int r = 0; r < p; ++r) rot_apply(g, G[(size_t)mp1 * r + k], G[(size_t)mp1 * r + i]);
                    rots.push_back(g);
                }
            }
            jend = j + 1;
            // residual estimate per right-hand side: rows nb .. nb + p of the rotated G
            bool done = true;
            for (int r = 0; r < p; ++r) {
                double e = 0.0;
                for (int i = nb; i < nb + p; ++i) e += std::norm(G[(size_t)mp1 * r + i]);
                done = done && (bnorm[r] == 0.0 || std::sqrt(e) / bnorm[r] < opts->tol);
            }
            if (opts->verbose) {
                double worst = 0.0;
                for (int r = 0; r < p; ++r) {
                    double e = 0.0;
                    for (int i = nb; i < nb + p; ++i) e += std::norm(G[(size_t)mp1 * r + i]);
                    worst = std::max(worst, bnorm[r] > 0.0 ? std::sqrt(e) / bnorm[r] : 0.0);
                }
                double el = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
                std::fprintf(stderr, "block gmres: %d products, worst estimated rel residual %.3e, %.1f s\n", iters,
                             worst, el);
                std::fflush(stderr);
            }
            if (done || iters >= opts->max_iter) break;
        }
        // Y = R^-1 G (upper triangular jend p), X_r += V Y_r
        const int nk = jend * p;
        for (int r = 0; r < p; ++r) {
            std::vector<cplx> y(nk, 0.0);
            for (int i = nk - 1; i >= 0; --i) {
                cplx acc = G[(size_t)mp1 * r + i];
                for (int k = i + 1; k < nk; ++k) acc -= H[(size_t)mp1 * k + i] * y[k];
                const cplx d = H[(size_t)mp1 * i + i];
                y[i] = std::abs(d) > 0.0 ? acc / d : cplx(0.0);
            }
            if ((rc = upload(y, nk))) return rc;
            launch_gemv_add(V, n, nk, h, X + r * n, n, s);
        }
    }
    for (int q = 0; q < p; ++q)
        if ((rc = scale_flat(c, X + q * n, xout + q * ld, 1))) return rc;
    if (hipStreamSynchronize(s) != hipSuccess) return IFS_E_HIP;
    const double secs = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    int all = 1;
    for (int q = 0; q < p; ++q) {
        if (info) {
            info[q].iterations = iters;
            info[q].converged = conv[q];
            info[q].rel_residual = bnorm[q] > 0.0 ? beta[q] / bnorm[q] : 0.0;
            info[q].seconds = secs;
            info[q].rel_residual_flat = flat[q];
        }
        all = all && conv[q];
    }
    return all ? IFS_OK : IFS_E_NOCONV;
}

// nrhs right-hand sides of one cluster in lock step (one system per column).
extern "C" int ifs_solve_batch_device(ifs_ctx *c, int32_t nrhs, const void *rhs_dev, void *x_dev, int64_t n,
                                      int64_t ld, const ifs_solve_opts *opts, ifs_solve_info *info) {
    if (!c || !rhs_dev || !x_dev || !opts || n != ifs_vector_length(c) || nrhs < 1 || ld < n) return IFS_E_ARG;
    if (check_opts(opts)) return IFS_E_ARG;
    Systems L;
    L.ncols = nrhs;
    L.ncol = n;
    for (int r = 0; r < nrhs; ++r) {
        L.col.push_back(r);
        L.off.push_back(0);
        L.len.push_back(n);
    }
    return solve_systems(c, L, (const double2 *)rhs_dev, (double2 *)x_dev, ld, opts, info);
}

// Every cluster of a multi-cluster context on its own Krylov space, all in one
// product per Arnoldi step (the operator is block diagonal).
extern "C" int ifs_solve_multi_device(ifs_ctx *c, const void *rhs_dev, void *x_dev, int64_t n,
                                      const ifs_solve_opts *opts, ifs_solve_info *info) {
    if (!c || !rhs_dev || !x_dev || !opts || n != ifs_vector_length(c)) return IFS_E_ARG;
    if (check_opts(opts)) return IFS_E_ARG;
    const int ng = ifs_cluster_count(c);
    std::vector<int64_t> first(ng + 1);
    ifs_cluster_offsets(c, nullptr, first.data());
    Systems L;
    L.ncols = 1;
    L.ncol = n;
    for (int g = 0; g < ng; ++g) {
        L.col.push_back(0);
        L.off.push_back(first[g]);
        L.len.push_back(first[g + 1] - first[g]);
    }
    return solve_systems(c, L, (const double2 *)rhs_dev, (double2 *)x_dev, n, opts, info);
}

// nrhs right-hand sides of one cluster by block GMRES (one shared Krylov space).
extern "C" int ifs_solve_block_device(ifs_ctx *c, int32_t nrhs, const void *rhs_dev, void *x_dev, int64_t n,
                                      int64_t ld, const ifs_solve_opts *opts, ifs_solve_info *info) {
    if (!c || !rhs_dev || !x_dev || !opts || n != ifs_vector_length(c) || nrhs < 1 || ld < n) return IFS_E_ARG;
    if (check_opts(opts)) return IFS_E_ARG;
    return solve_block(c, nrhs, (const double2 *)rhs_dev, (double2 *)x_dev, ld, opts, info);
}

extern "C" int ifs_solve_block(ifs_ctx *c, int32_t nrhs, const double *rhs, double *x, int64_t n,
                               const ifs_solve_opts *opts, ifs_solve_info *info) {
    if (!c || !rhs || !x || !opts || n != ifs_vector_length(c) || nrhs < 1) return IFS_E_ARG;
    hipStream_t s = ctx_stream(c);
    DevBuf db, dx;
    int rc;
    if ((rc = db.alloc(16ull * n * nrhs)) || (rc = dx.alloc(16ull * n * nrhs))) return rc;
    if (hipMemcpyAsync(db.p, rhs, 16ull * n * nrhs, hipMemcpyHostToDevice, s) != hipSuccess ||
        (opts->use_x0 && hipMemcpyAsync(dx.p, x, 16ull * n * nrhs, hipMemcpyHostToDevice, s) != hipSuccess))
        return IFS_E_HIP;
    rc = ifs_solve_block_device(c, nrhs, db.p, dx.p, n, n, opts, info);
    if (rc == IFS_OK || rc == IFS_E_NOCONV || rc == IFS_E_BREAKDOWN) {
        if (hipMemcpyAsync(x, dx.p, 16ull * n * nrhs, hipMemcpyDeviceToHost, s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess)
            return IFS_E_HIP;
    }
    return rc;
}

extern "C" int ifs_solve_multi(ifs_ctx *c, const double *rhs, double *x, int64_t n, const ifs_solve_opts *opts,
                               ifs_solve_info *info) {
    if (!c || !rhs || !x || !opts || n != ifs_vector_length(c)) return IFS_E_ARG;
    hipStream_t s = ctx_stream(c);
    DevBuf db, dx;
    int rc;
    if ((rc = db.alloc(16ull * n)) || (rc = dx.alloc(16ull * n))) return rc;
    if (hipMemcpyAsync(db.p, rhs, 16ull * n, hipMemcpyHostToDevice, s) != hipSuccess ||
        (opts->use_x0 && hipMemcpyAsync(dx.p, x, 16ull * n, hipMemcpyHostToDevice, s) != hipSuccess))
        return IFS_E_HIP;
    rc = ifs_solve_multi_device(c, db.p, dx.p, n, opts, info);
    if (rc == IFS_OK || rc == IFS_E_NOCONV || rc == IFS_E_BREAKDOWN) {
        if (hipMemcpyAsync(x, dx.p, 16ull * n, hipMemcpyDeviceToHost, s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess)
            return IFS_E_HIP;
    }
    return rc;
}

extern "C" int ifs_solve_batch(ifs_ctx *c, int32_t nrhs, const double *rhs, double *x, int64_t n,
                               const ifs_solve_opts *opts, ifs_solve_info *info) {
    if (!c || !rhs || !x || !opts || n != ifs_vector_length(c) || nrhs < 1) return IFS_E_ARG;
    hipStream_t s = ctx_stream(c);
    DevBuf db, dx;
    int rc;
    if ((rc = db.alloc(16ull * n * nrhs)) || (rc = dx.alloc(16ull * n * nrhs))) return rc;
    if (hipMemcpyAsync(db.p, rhs, 16ull * n * nrhs, hipMemcpyHostToDevice, s) != hipSuccess ||
        (opts->use_x0 && hipMemcpyAsync(dx.p, x, 16ull * n * nrhs, hipMemcpyHostToDevice, s) != hipSuccess))
        return IFS_E_HIP;
    rc = ifs_solve_batch_device(c, nrhs, db.p, dx.p, n, n, opts, info);
    if (rc == IFS_OK || rc == IFS_E_NOCONV || rc == IFS_E_BREAKDOWN) {
        if (hipMemcpyAsync(x, dx.p, 16ull * n * nrhs, hipMemcpyDeviceToHost, s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess)
            return IFS_E_HIP;
    }
    return rc;
}

extern "C" int ifs_solve(ifs_ctx *c, const double *rhs, double *x, int64_t n, const ifs_solve_opts *opts,
                         ifs_solve_info *info) {
    if (!c || !rhs || !x || !opts || n != ifs_vector_length(c)) return IFS_E_ARG;
    hipStream_t s = ctx_stream(c);
    void *db = nullptr, *dx = nullptr;
    if (hipMalloc(&db, 16ull * n) != hipSuccess) return IFS_E_NOMEM;
    if (hipMalloc(&dx, 16ull * n) != hipSuccess) {
        (void)hipFree(db);
        return IFS_E_NOMEM;
    }
    int rc = IFS_OK;
    if (hipMemcpyAsync(db, rhs, 16ull * n, hipMemcpyHostToDevice, s) != hipSuccess ||
        (opts->use_x0 && hipMemcpyAsync(dx, x, 16ull * n, hipMemcpyHostToDevice, s) != hipSuccess))
        rc = IFS_E_HIP;
    if (!rc) rc = ifs_solve_device(c, db, dx, n, opts, info);
    if (rc == IFS_OK || rc == IFS_E_NOCONV || rc == IFS_E_BREAKDOWN) {
        if (hipMemcpyAsync(x, dx, 16ull * n, hipMemcpyDeviceToHost, s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess)
            rc = IFS_E_HIP;
    }
    (void)hipFree(db);
    (void)hipFree(dx);
    return rc;
}

// x-polarised plane wave along +z: p_{n,+-1}, q_{n,+-1} from the closed forms of
// pi_mn, tau_mn at cos(alpha) = 1 (libmath/src/math/lib_math_legendre.f90:834-962,
// Condon-Shortley phase removed for odd |m|) in
// p = tau_mn e^{-i m beta} e^{i k.d} / (n(n+1)),  q = pi_mn e^{-i m beta} e^{i k.d} / (n(n+1))
// (FoggySim/src/lib/mie_theory/lib_mie_illumination.f90:295-354, :636-763),
// then rhs = (a_n p, b_n q) (lib_mie_ms_solver_interface.f90:230-315).
extern "C" int ifs_plane_wave_rhs(ifs_ctx *c, double *rhs, int64_t n) {
    if (!c || !rhs || n != ifs_vector_length(c)) return IFS_E_ARG;
    const int ns = ctx_ns(c), N = ctx_N(c);
    const double k = ctx_k(c);
    const double *pos = ctx_pos(c);
    std::vector<cplx> an((size_t)ns * N), bn((size_t)ns * N);
    int rc = ifs_get_mie(c, (double *)an.data(), (double *)bn.data());
    if (rc) return rc;
    cplx *out = (cplx *)rhs;
    const int64_t blk = (int64_t)N * (N + 2);
    for (int64_t i = 0; i < n; ++i) out[i] = 0.0;
    for (int j = 0; j < ns; ++j) {
        cplx ph = std::exp(cplx(0.0, k * pos[3 * j + 2]));
        for (int nn = 1; nn <= N; ++nn) {
            double inv = 1.0 / (nn * (nn + 1.0));
            double pi_p = nn * (nn + 1.0) / 2.0, pi_m = 0.5;
            double tau_p = nn * (nn + 1.0) / 2.0, tau_m = -0.5;
            cplx pp = ph * tau_p * inv, pm = ph * tau_m * inv;
            cplx qp = ph * pi_p * inv, qm = ph * pi_m * inv;
            int64_t o = (int64_t)j * 2 * blk;
            int64_t ip = nn * nn - 1 + 1 + nn, im = nn * nn - 1 - 1 + nn;
            out[o + ip] = an[(size_t)j * N + nn - 1] * pp;
            out[o + im] = an[(size_t)j * N + nn - 1] * pm;
            out[o + blk + ip] = bn[(size_t)j * N + nn - 1] * qp;
            out[o + blk + im] = bn[(size_t)j * N + nn - 1] * qm;
        }
    }
    return IFS_OK;
}
