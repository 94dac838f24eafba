// Optics of a solved cluster (gfx950): plane-wave expansion coefficients, far
// field, amplitude and Mueller matrices, cross sections.
//
// Conventions (Xu's, as the reference's Mie code uses them):
//   incident wave along (alpha, beta), amplitude 1, at sphere centre d_j
//     p_mn = e^{i k khat.d_j} tau_mn(alpha) e^{-i m beta} / (n(n+1)),  q_mn likewise with pi_mn
//     (FoggySim/src/lib/mie_theory/lib_mie_illumination.f90:636-763);
//   far field E_s ~ e^{ikr}/(kr) F, with, in the normalised basis c_hat = s_nm c,
//     F_theta =  i sum_j e^{-ik rhat.d_j} sum_nm e^{i m phi} (a_hat T_nm + b_hat P_nm)
//     F_phi   = -  sum_j e^{-ik rhat.d_j} sum_nm e^{i m phi} (a_hat P_nm + b_hat T_nm)
//   where T_nm = s_nm tau_mn / (n(n+1)) and P_nm = s_nm pi_mn / (n(n+1)) are, through
//   the Wigner functions d^n_{m,+-1}(theta),
//     T_nm = (-1)^{m+1} sqrt(2n+1) (d^n_{m,1} - d^n_{m,-1}) / 2
//     P_nm = (-1)^{m+1} sqrt(2n+1) (d^n_{m,1} + d^n_{m,-1}) / 2   (bounded for every n);
//   cross sections (lib_mie_ss_helper_functions.f90:1380-1460, Xu eq. 57, summed over
//   the spheres; absorption from each sphere's exciting field a^j_mn / a_n^j):
//     C_ext = 4 pi/k^2 sum Re(conj(p_hat) a_hat + conj(q_hat) b_hat)
//     C_abs = 4 pi/k^2 sum |a_hat|^2 (Re(1/a_n) - 1) + |b_hat|^2 (Re(1/b_n) - 1),
//     C_sca = C_ext - C_abs.
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>
#include <cmath>
#include <complex>
#include <map>
#include <mutex>
#include <vector>

#include "ifs_engine.h"
#include "ifs_wigner.h"

namespace ifs {

namespace {

__device__ __forceinline__ double2 cmul_(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// T_nm, P_nm at the polar angles theta[i]: tab[i * N(N+2) + fidx(n,m)] = (T, P).
// One thread per order m >= 0 and FFT directions, running the recurrences of d^n_{m,1}
// and d^n_{m,-1} upward in n; the square roots and the division of a step and the
// log-gammas of the seeds serve all FFT directions, and
//   T_{n,-m} = (-1)^m T_nm,  P_{n,-m} = -(-1)^m P_nm
// the negative orders.  Bound by the FP64 chain of the recurrences (6516 directions of order
// 22: 57 us; 92 us with a thread per signed order and direction).
constexpr int FFT = 4;
__global__ __launch_bounds__(256) void k_ff_tables(int N, int ndir, const double *__restrict__ theta,
                                                   double2 *__restrict__ tab) {
    const int mw = min(N + 1, 256), subs = 256 / mw, sub = threadIdx.x / mw;
    if (sub >= subs) return;
    const int i0 = (blockIdx.x * subs + sub) * FFT;
    if (i0 >= ndir) return;
    const int64_t blk = (int64_t)N * (N + 2);
    double cb[FFT], ch[FFT], sh[FFT];
#pragma unroll
    for (int d = 0; d < FFT; ++d) {
        const double th = theta[min(i0 + d, ndir - 1)];
        cb[d] = cos(th);
        ch[d] = cos(0.5 * th);
        sh[d] = sin(0.5 * th);
    }
    for (int m = threadIdx.x % mw; m <= N; m += mw) {
        const int n0 = m > 1 ? m : 1;
        const double sm = (m & 1) ? -1.0 : 1.0;  // (-1)^m
        const double lp = wigner_seed_ln(m, 1), lq = wigner_seed_ln(m, -1);
        double p1[FFT], p2[FFT], q1[FFT], q2[FFT];
#pragma unroll
        for (int d = 0; d < FFT; ++d) {
            p1[d] = wigner_seed(m, 1, ch[d], sh[d], lp);
            q1[d] = wigner_seed(m, -1, ch[d], sh[d], lq);
            p2[d] = q2[d] = 0.0;
        }
        for (int n = n0; n <= N; ++n) {
            if (n > n0) {
                const double nn = n, o = nn - 1.0, m2 = (double)m * m;
                const double inv = 1.0 / (o * sqrt((nn * nn - m2) * (nn * nn - 1.0)));
                const double F = (2.0 * nn - 1.0) * inv, G = nn * sqrt((o * o - m2) * (o * o - 1.0)) * inv;
#pragma unroll
                for (int d = 0; d < FFT; ++d) {
                    const double pn = F * (nn * o * cb[d] - m) * p1[d] - G * p2[d];
                    const double qn = F * (nn * o * cb[d] + m) * q1[d] - G * q2[d];
                    p2[d] = p1[d];
                    p1[d] = pn;
                    q2[d] = q1[d];
                    q1[d] = qn;
                }
            }
            const double f = -0.5 * sm * sqrt(2.0 * n + 1.0);
#pragma unroll
            for (int d = 0; d < FFT; ++d) {
                if (i0 + d >= ndir) break;
                const double T = f * (p1[d] - q1[d]), P = f * (p1[d] + q1[d]);
                double2 *o = tab + (int64_t)(i0 + d) * blk + (int64_t)n * n - 1 + n;
                o[m] = make_double2(T, P);
                if (m > 0) o[-m] = make_double2(sm * T, -sm * P);
            }
        }
    }
}

// The sum over spheres first: for every entry e = (n, m),
//   Y_a[d, e] = sum_j e^{-ik rhat_d.d_j} a_j[e]   (and Y_b), a complex matrix product of the
// phases [directions x spheres] with the coefficients [spheres x entries], in FP64 MFMA
// (16 directions x 16 entries x 4 spheres a step, a and b with the same phases); then the
// contraction with T, P, s_nm and e^{i m phi} once per (d, e) instead of once per
// (d, e, sphere): 16 instead of about 30 flops per (d, e, sphere), and the phases and
// coefficients of a step serve 16 directions.
// A block: 16 directions, the phases of FFC spheres at a time in LDS; its waves share out
// the entries in tiles of 16, strided by all waves of the directions' blocks (gridDim.y of
// them).  Spheres come in descending order L_j, so a tile of degrees >= n ends its product
// at the first sphere with L_j < n.  Coefficients beyond a sphere's L_j are not read.
// out[(blockIdx.y * ndir + i) * 2 + {0, 1}]: this block's part of (F_theta, F_phi).
// 200 spheres of orders up to 22, 6516 directions: 224 us (6.5 GFLOP in the matrix cores, 90 us
// at their rate; the rest the phases' sincos, the contraction and the first loads of a tile)
// against 1641 us with a thread per entry and sphere.  Two tiles of directions a wave, for
// half the coefficient reads: 252 us, so those do not bound it.
constexpr int FFC = 128;  // spheres per chunk of phases
constexpr int FFE = 112;  // orders up to which e^{i m phi} is kept in LDS: 64 KB with the phases
typedef double ffv4 __attribute__((ext_vector_type(4)));

template <bool EM>
__global__ __launch_bounds__(256, EM ? 3 : 2) void k_far_field(
    int N, int ns, const int32_t *__restrict__ Leff, const int32_t *__restrict__ order,
                                                   const double *__restrict__ pos, double k,
                                                   const double *__restrict__ snm, const double2 *__restrict__ x,
                                                   int ndir, const double *__restrict__ theta,
                                                   const double *__restrict__ phi, const double2 *__restrict__ tab,
                                                   double2 *__restrict__ out) {
    extern __shared__ double2 em[];  // EM: [16][N + 1], e^{i m phi}
    __shared__ double2 ph[FFC * 16];  // [sphere][direction]
    __shared__ int2 sp[FFC];           // (sphere, entries of a block)
    __shared__ double rh[16][3];
    __shared__ double2 red[4][16][2];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, col = lane & 15, lk = lane >> 4;
    const int i0 = blockIdx.x * 16;
    const int64_t blk = (int64_t)N * (N + 2);
    const int nt = (int)((blk + 15) / 16);
    if (EM)
        for (int q = tid; q < 16 * (N + 1); q += 256) {
            const int d = q / (N + 1), m = q % (N + 1);
            double s, c;
            sincos((double)m * phi[min(i0 + d, ndir - 1)], &s, &c);
            em[q] = make_double2(c, s);
        }
    if (tid < 16) {
        const int i = min(i0 + tid, ndir - 1);
        const double t = theta[i], f = phi[i];
        rh[tid][0] = sin(t) * cos(f);
        rh[tid][1] = sin(t) * sin(f);
        rh[tid][2] = cos(t);
    }
    double2 ft[4] = {}, fp[4] = {};
    for (int j0 = 0; j0 < ns; j0 += FFC) {
        const int jn = min(FFC, ns - j0), jp = (jn + 3) & ~3;
        __syncthreads();
        for (int q = tid; q < jp; q += 256) {
            int2 v = make_int2(0, 0);
            if (q < jn) {
                v.x = order[j0 + q];
                const int L = Leff[v.x];
                v.y = L * (L + 2);
            }
            sp[q] = v;
        }
        for (int q = tid; q < jp * 16; q += 256) {
            const int j = q >> 4, d = q & 15;
            double2 v = make_double2(0.0, 0.0);
            if (j < jn) {
                const double *p = pos + 3 * (int64_t)order[j0 + j];
                const double arg = -k * (rh[d][0] * p[0] + rh[d][1] * p[1] + rh[d][2] * p[2]);
                sincos(arg, &v.y, &v.x);
            }
            ph[q] = v;
        }
        __syncthreads();
        for (int t = blockIdx.y * 4 + wave; t < nt; t += gridDim.y * 4) {
            const int e = t * 16 + col;
            ffv4 ar = {}, ai = {}, br = {}, bi = {};
            int je = 0;  // spheres that hold any entry of this tile
            for (int lo = jn; lo > 0; lo >>= 1)
                while (je + lo <= jn && __builtin_amdgcn_readfirstlane(sp[je + lo - 1].y) > t * 16) je += lo;
            auto load = [&](int j, double2 &a, double2 &b) {
                const int2 s = sp[j + lk];
                a = b = make_double2(0.0, 0.0);
                if (e < s.y) {
                    const double2 *xa = x + (int64_t)s.x * 2 * blk + e;
                    a = xa[0];
                    b = xa[blk];
                }
            };
            double2 an, bn;
            if (je > 0) load(0, an, bn);
            for (int j = 0; j < je; j += 4) {
                const double2 a = an, b = bn;
                if (j + 4 < je) load(j + 4, an, bn);
                const double2 f = ph[(j + lk) * 16 + col];
                ar = __builtin_amdgcn_mfma_f64_16x16x4f64(f.x, a.x, ar, 0, 0, 0);
                ai = __builtin_amdgcn_mfma_f64_16x16x4f64(f.x, a.y, ai, 0, 0, 0);
                br = __builtin_amdgcn_mfma_f64_16x16x4f64(f.x, b.x, br, 0, 0, 0);
                bi = __builtin_amdgcn_mfma_f64_16x16x4f64(f.x, b.y, bi, 0, 0, 0);
                ar = __builtin_amdgcn_mfma_f64_16x16x4f64(-f.y, a.y, ar, 0, 0, 0);
                ai = __builtin_amdgcn_mfma_f64_16x16x4f64(f.y, a.x, ai, 0, 0, 0);
                br = __builtin_amdgcn_mfma_f64_16x16x4f64(-f.y, b.y, br, 0, 0, 0);
                bi = __builtin_amdgcn_mfma_f64_16x16x4f64(f.y, b.x, bi, 0, 0, 0);
            }
            if (e >= blk) continue;
            int n = (int)sqrt((double)(e + 1));
            while ((n + 1) * (n + 1) - 1 <= e) ++n;
            while (n * n - 1 > e) --n;
            const int m = e - (n * n - 1) - n, am = m < 0 ? -m : m;
            const double s = snm[e];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int d = 4 * v + lk, i = min(i0 + d, ndir - 1);
                double2 w;
                if (EM)
                    w = em[d * (N + 1) + am];
                else
                    sincos((double)am * phi[i], &w.y, &w.x);
                if (m < 0) w.y = -w.y;
                const double2 tp = tab[(int64_t)i * blk + e];  // (T, P)
                const double2 a = make_double2(s * ar[v], s * ai[v]), b = make_double2(s * br[v], s * bi[v]);
                const double2 vt = cmul_(w, make_double2(a.x * tp.x + b.x * tp.y, a.y * tp.x + b.y * tp.y));
                const double2 vp = cmul_(w, make_double2(a.x * tp.y + b.x * tp.x, a.y * tp.y + b.y * tp.x));
                ft[v].x += vt.x;
                ft[v].y += vt.y;
                fp[v].x += vp.x;
                fp[v].y += vp.y;
            }
        }
    }
    // over the 16 entries' lanes, then over the waves (fixed order)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        for (int o = 8; o > 0; o >>= 1) {
            ft[v].x += __shfl_xor(ft[v].x, o);
            ft[v].y += __shfl_xor(ft[v].y, o);
            fp[v].x += __shfl_xor(fp[v].x, o);
            fp[v].y += __shfl_xor(fp[v].y, o);
        }
        if (col == 0) {
            red[wave][4 * v + lk][0] = ft[v];
            red[wave][4 * v + lk][1] = fp[v];
        }
    }
    __syncthreads();
    if (tid < 32 && i0 + (tid >> 1) < ndir) {
        const int d = tid >> 1, c = tid & 1;
        double2 s = red[0][d][c];
        for (int w = 1; w < 4; ++w) {
            s.x += red[w][d][c].x;
            s.y += red[w][d][c].y;
        }
        // F_theta = i * sum, F_phi = - sum
        out[((int64_t)blockIdx.y * ndir + i0 + d) * 2 + c] = c == 0 ? make_double2(-s.y, s.x) : make_double2(-s.x, -s.y);
    }
}

// out[q] = sum over the parts of part[g * n + q]
__global__ void k_ff_sum(int64_t n, int parts, const double2 *__restrict__ part, double2 *__restrict__ out) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    double2 s = part[q];
    for (int g = 1; g < parts; ++g) {
        s.x += part[g * n + q].x;
        s.y += part[g * n + q].y;
    }
    out[q] = s;
}

// Blocks that share 16 directions' entries, at most `room` for their parts of the sums:
// enough for 1024 blocks, each with a tile for
// every wave (6516 directions: 224 us; for 512 blocks 262, for 2048 235).
int ff_parts(int N, int ndir, int64_t room) {
    const int64_t rows = (ndir + 15) / 16, nt = ((int64_t)N * (N + 2) + 15) / 16;
    int64_t g = std::min<int64_t>((1024 + rows - 1) / rows, (nt + 3) / 4);
    g = std::min<int64_t>(g, room / (2 * (int64_t)ndir));
    return (int)std::max<int64_t>(1, g);
}

// tab: ndir * N(N+2) entries, then 2 ndir per part where there is more than one
int ff_launch(ifs_ctx *c, const void *x, int ndir, const double *theta, const double *phi, double2 *tab, int parts,
              double2 *out) {
    const int N = c->N, per = 256 / std::min(N + 1, 256) * FFT;
    double2 *dst = parts > 1 ? tab + (int64_t)ndir * N * (N + 2) : out;
    hipLaunchKernelGGL(k_ff_tables, dim3((ndir + per - 1) / per), dim3(256), 0, c->stream, N, ndir, theta, tab);
    const int32_t *Leff = c->d_Leff.as<int32_t>();
    const bool em = N <= FFE;
    auto far = em ? k_far_field<true> : k_far_field<false>;
    hipLaunchKernelGGL(far, dim3((ndir + 15) / 16, parts), dim3(256), em ? sizeof(double2) * 16 * (N + 1) : 0,
                       c->stream, N, c->ns, Leff, Leff + c->ns,
                       c->d_pos.as<double>(), c->prm.k, c->d_snm.as<double>(), (const double2 *)x, ndir, theta, phi,
                       tab, dst);
    if (parts > 1)
        hipLaunchKernelGGL(k_ff_sum, dim3((unsigned)((2 * (int64_t)ndir + 255) / 256)), dim3(256), 0, c->stream,
                           2 * (int64_t)ndir, parts, dst, out);
    return hipGetLastError() == hipSuccess ? IFS_OK : IFS_E_HIP;
}

// Per-sphere partial sums for the cross sections: part[j] = (extinction, absorption)
// sums (without the 4 pi / k^2 factor).
__global__ __launch_bounds__(256) void k_xsec(int N, const int32_t *__restrict__ Leff, const double *__restrict__ snm,
                                              const double2 *__restrict__ x, const double2 *__restrict__ p,
                                              const double2 *__restrict__ an, const double2 *__restrict__ bn,
                                              double2 *__restrict__ part) {
    __shared__ double2 red[256];
    const int j = blockIdx.x;
    const int L = Leff[j];
    const int cnt = L * (L + 2);
    const int64_t blk = (int64_t)N * (N + 2);
    const double2 *xa = x + (int64_t)j * 2 * blk;
    const double2 *pa = p + (int64_t)j * 2 * blk;
    double ext = 0.0, abs_ = 0.0;
    for (int e = threadIdx.x; e < cnt; e += blockDim.x) {
        int n = (int)sqrt((double)(e + 1));
        while ((n + 1) * (n + 1) - 1 <= e) ++n;
        while (n * n - 1 > e) --n;
        const double s2 = snm[e] * snm[e];
        const double2 a = xa[e], b = xa[e + blk], pp = pa[e], qq = pa[e + blk];
        ext += s2 * (pp.x * a.x + pp.y * a.y + qq.x * b.x + qq.y * b.y);
        const double2 A = an[(int64_t)j * N + n - 1], B = bn[(int64_t)j * N + n - 1];
        const double na = A.x * A.x + A.y * A.y, nb = B.x * B.x + B.y * B.y;
        // Re(1/a_n) - 1 = Re(a_n)/|a_n|^2 - 1
        if (na > 0.0) abs_ += s2 * (a.x * a.x + a.y * a.y) * (A.x / na - 1.0);
        if (nb > 0.0) abs_ += s2 * (b.x * b.x + b.y * b.y) * (B.x / nb - 1.0);
    }
    red[threadIdx.x] = make_double2(ext, abs_);
    __syncthreads();
    for (int h = blockDim.x / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) {
            red[threadIdx.x].x += red[threadIdx.x + h].x;
            red[threadIdx.x].y += red[threadIdx.x + h].y;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) part[j] = red[0];
}

// Host: d^n_{m,+-1}(beta) for n = 1..N, |m| <= n, in long double (seed in logs,
// three-term recurrence in n); dp/dm indexed at n*n-1+m+n.
void d_pm1_host(int N, long double beta, std::vector<long double> &dp, std::vector<long double> &dm) {
    const int64_t blk = (int64_t)N * (N + 2);
    dp.assign(blk, 0.0L);
    dm.assign(blk, 0.0L);
    const long double cb = cosl(beta), c = cosl(0.5L * beta), s = sinl(0.5L * beta);
    auto seed = [&](int k, int m) -> long double {
        long double sign = 1.0L;
        if (std::abs(k) < std::abs(m)) {
            std::swap(k, m);
            if ((k - m) & 1) sign = -sign;
        }
        int j = std::abs(k), ec, es;
        if (k >= 0) {
            ec = j + m;
            es = j - m;
            if (es & 1) sign = -sign;
        } else {
            ec = j - m;
            es = j + m;
        }
        long double lv = 0.5L * (lgammal(2.0L * j + 1.0L) - lgammal((long double)(j + m) + 1.0L) -
                                 lgammal((long double)(j - m) + 1.0L));
        if (ec > 0) {
            if (c <= 0.0L) return 0.0L;
            lv += ec * logl(c);
        }
        if (es > 0) {
            if (s <= 0.0L) return 0.0L;
            lv += es * logl(s);
        }
        return sign * expl(lv);
    };
    auto step = [&](int n, int k, int m, long double d1, long double d2) {
        long double nn = n, k2 = (long double)k * k, m2 = (long double)m * m;
        long double num = (2.0L * nn - 1.0L) * (nn * (nn - 1.0L) * cb - (long double)k * m) * d1 -
                          nn * sqrtl(((nn - 1) * (nn - 1) - k2) * ((nn - 1) * (nn - 1) - m2)) * d2;
        long double den = (nn - 1.0L) * sqrtl((nn * nn - k2) * (nn * nn - m2));
        return num / den;
    };
    for (int m = -N; m <= N; ++m) {
        const int n0 = std::max(std::abs(m), 1);
        long double p1 = seed(m, 1), q1 = seed(m, -1), p2 = 0.0L, q2 = 0.0L;
        for (int n = n0; n <= N; ++n) {
            if (n > n0) {
                long double pn = step(n, m, 1, p1, p2), qn = step(n, m, -1, q1, q2);
                p2 = p1;
                p1 = pn;
                q2 = q1;
                q1 = qn;
            }
            dp[n * n - 1 + m + n] = p1;
            dm[n * n - 1 + m + n] = q1;
        }
    }
}

}  // namespace

}  // namespace ifs

// Scratch of ifs_far_field_device_noalloc: the per-direction T/P tables and,
// as far as there is room, parts of the sums, in a fixed array of this library on every GPU it runs on (held until the process
// ends).  Host code never uses the array's name as an address: its device address
// is looked up once per device (far_field_scratch) and passed to the kernels.
static __device__ __align__(256) double2 scratch[IFS_FF_SCRATCH_ENTRIES];

namespace ifs {
int far_field_scratch(int device, void **out) {
    static std::mutex mu;
    static std::map<int, void *> per_device;
    std::lock_guard<std::mutex> lock(mu);
    auto it = per_device.find(device);
    if (it != per_device.end()) {
        *out = it->second;
        return IFS_OK;
    }
    void *p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || p == nullptr) return IFS_E_HIP;
    per_device[device] = p;
    *out = p;
    return IFS_OK;
}
}  // namespace ifs

using cplx = std::complex<double>;

extern "C" int ifs_plane_wave(ifs_ctx *c, double alpha, double beta, double *p_out, int64_t n) {
    if (!c || !p_out || n != ifs_vector_length(c)) return IFS_E_ARG;
    const int N = c->N, ns = c->ns;
    const int64_t blk = (int64_t)N * (N + 2);
    std::vector<long double> dp, dm;
    ifs::d_pm1_host(N, (long double)alpha, dp, dm);
    // angular part tau_mn / (n(n+1)) and pi_mn / (n(n+1)) (flat layout, unnormalised)
    std::vector<cplx> ta(blk), pa(blk);
    for (int nn = 1; nn <= N; ++nn)
        for (int m = -nn; m <= nn; ++m) {
            int64_t e = (int64_t)nn * nn - 1 + m + nn;
            // s_nm = sqrt(n(n+1)(2n+1)(n-m)!/(n+m)!)
            long double ls = 0.5L * (logl((long double)nn * (nn + 1) * (2 * nn + 1)) + lgammal(nn - m + 1.0L) -
                                     lgammal(nn + m + 1.0L));
            long double sg = (std::abs(m) & 1) ? 1.0L : -1.0L;  // (-1)^{m+1}
            long double f = 0.5L * sg * sqrtl(2.0L * nn + 1.0L) / expl(ls);
            long double t = f * (dp[e] - dm[e]), p = f * (dp[e] + dm[e]);
            long double a = -(long double)m * beta;
            cplx em((double)cosl(a), (double)sinl(a));
            ta[e] = (double)t * em;
            pa[e] = (double)p * em;
        }
    const double kh[3] = {std::sin(alpha) * std::cos(beta), std::sin(alpha) * std::sin(beta), std::cos(alpha)};
    cplx *out = (cplx *)p_out;
    for (int j = 0; j < ns; ++j) {
        double kd = c->prm.k * (kh[0] * c->pos[3 * j] + kh[1] * c->pos[3 * j + 1] + kh[2] * c->pos[3 * j + 2]);
        cplx ph(std::cos(kd), std::sin(kd));
        for (int64_t e = 0; e < blk; ++e) {
            out[(int64_t)j * 2 * blk + e] = ph * ta[e];
            out[(int64_t)j * 2 * blk + blk + e] = ph * pa[e];
        }
    }
    return IFS_OK;
}

// TE mode of the reference's illumination: the TM coefficients with p and q exchanged
// (lib_mie_illumination.f90:347-352; the polarisation turned by 90 degrees about the
// propagation direction).
extern "C" int ifs_plane_wave_mode(ifs_ctx *c, double alpha, double beta, int32_t te, double *p_out, int64_t n) {
    if (te != 0 && te != 1) return IFS_E_ARG;
    int rc = ifs_plane_wave(c, alpha, beta, p_out, n);
    if (rc || !te) return rc;
    const int64_t blk = (int64_t)c->N * (c->N + 2);
    cplx *out = (cplx *)p_out;
    for (int j = 0; j < c->ns; ++j)
        for (int64_t e = 0; e < blk; ++e) std::swap(out[(int64_t)j * 2 * blk + e], out[(int64_t)j * 2 * blk + blk + e]);
    return IFS_OK;
}

extern "C" int ifs_plane_wave_rhs_dir(ifs_ctx *c, double alpha, double beta, double *rhs, int64_t n) {
    return ifs_plane_wave_rhs_mode(c, alpha, beta, 0, rhs, n);
}

extern "C" int ifs_plane_wave_rhs_mode(ifs_ctx *c, double alpha, double beta, int32_t te, double *rhs, int64_t n) {
    int rc = ifs_plane_wave_mode(c, alpha, beta, te, rhs, n);
    if (rc) return rc;
    const int N = c->N, ns = c->ns;
    const int64_t blk = (int64_t)N * (N + 2);
    std::vector<cplx> an((size_t)ns * N), bn((size_t)ns * N);
    if ((rc = ifs_get_mie(c, (double *)an.data(), (double *)bn.data()))) return rc;
    cplx *out = (cplx *)rhs;
    for (int j = 0; j < ns; ++j)
        for (int nn = 1; nn <= N; ++nn)
            for (int m = -nn; m <= nn; ++m) {
                int64_t e = (int64_t)nn * nn - 1 + m + nn;
                bool keep = nn <= c->Leff[j] && c->active[j];
                out[(int64_t)j * 2 * blk + e] *= keep ? an[(size_t)j * N + nn - 1] : 0.0;
                out[(int64_t)j * 2 * blk + blk + e] *= keep ? bn[(size_t)j * N + nn - 1] : 0.0;
            }
    return IFS_OK;
}

extern "C" int ifs_cross_sections_device(ifs_ctx *c, const void *x_dev, const void *p_dev, int64_t n,
                                         double out[3]) {
    if (!c || !x_dev || !p_dev || !out || n != ifs_vector_length(c)) return IFS_E_ARG;
    ifs::DevBuf part;
    int rc;
    if ((rc = part.alloc(16ull * c->ns))) return rc;
    hipLaunchKernelGGL(ifs::k_xsec, dim3(c->ns), dim3(256), 0, c->stream, c->N, c->d_Leff.as<int32_t>(),
                       c->d_snm.as<double>(), (const double2 *)x_dev, (const double2 *)p_dev,
                       c->d_an.as<double2>(), c->d_bn.as<double2>(), part.as<double2>());
    if (hipGetLastError() != hipSuccess) return IFS_E_HIP;
    std::vector<double2> h(c->ns);
    if (hipMemcpyAsync(h.data(), part.p, 16ull * c->ns, hipMemcpyDeviceToHost, c->stream) != hipSuccess ||
        hipStreamSynchronize(c->stream) != hipSuccess)
        return IFS_E_HIP;
    double ext = 0.0, ab = 0.0;
    for (int j = 0; j < c->ns; ++j) {
        ext += h[j].x;
        ab += h[j].y;
    }
    const double f = 4.0 * M_PI / (c->prm.k * c->prm.k);
    out[0] = f * (ext - ab);
    out[1] = f * ext;
    out[2] = f * ab;
    return IFS_OK;
}

extern "C" int ifs_cross_sections(ifs_ctx *c, const double *x, const double *p, int64_t n, double out[3]) {
    if (!c || !x || !p || !out || n != ifs_vector_length(c)) return IFS_E_ARG;
    ifs::DevBuf dx, dp;
    int rc;
    if ((rc = dx.alloc(16ull * n)) || (rc = dp.alloc(16ull * n))) return rc;
    if (hipMemcpy(dx.p, x, 16ull * n, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dp.p, p, 16ull * n, hipMemcpyHostToDevice) != hipSuccess)
        return IFS_E_HIP;
    return ifs_cross_sections_device(c, dx.p, dp.p, n, out);
}

extern "C" int ifs_far_field_device(ifs_ctx *c, const void *x_dev, int64_t n, int32_t ndir, const void *theta_dev,
                                    const void *phi_dev, void *out_dev) {
    if (!c || !x_dev || !theta_dev || !phi_dev || !out_dev || n != ifs_vector_length(c) || ndir < 0)
        return IFS_E_ARG;
    if (ndir == 0) return IFS_OK;
    const int64_t entries = (int64_t)ndir * c->N * (c->N + 2);
    const int parts = ifs::ff_parts(c->N, ndir, INT64_MAX);
    int rc;
    ifs::DevBuf tab;
    if ((rc = tab.alloc(16ull * (entries + 2ll * ndir * (parts > 1 ? parts : 0))))) return rc;
    if ((rc = ifs::ff_launch(c, x_dev, ndir, (const double *)theta_dev, (const double *)phi_dev, tab.as<double2>(),
                             parts, (double2 *)out_dev)))
        return rc;
    if (hipStreamSynchronize(c->stream) != hipSuccess) return IFS_E_HIP;  // tab is freed on return
    return IFS_OK;
}

extern "C" int ifs_far_field_device_noalloc(ifs_ctx *c, const void *x_dev, int64_t n, int32_t ndir,
                                            const void *theta_dev, const void *phi_dev, void *out_dev) {
    if (!c || !x_dev || !theta_dev || !phi_dev || !out_dev || n != ifs_vector_length(c) || ndir < 0)
        return IFS_E_ARG;
    if (ndir == 0) return IFS_OK;
    const int64_t entries = (int64_t)ndir * c->N * (c->N + 2);
    if (entries > (int64_t)IFS_FF_SCRATCH_ENTRIES) return IFS_E_ARG;
    if (!c->ff_scratch || !c->d_pos.p) return IFS_E_ARG;
    // every entry that a kernel reads of the scratch array is written first
    return ifs::ff_launch(c, x_dev, ndir, (const double *)theta_dev, (const double *)phi_dev,
                          (double2 *)c->ff_scratch,
                          ifs::ff_parts(c->N, ndir, (int64_t)IFS_FF_SCRATCH_ENTRIES - entries), (double2 *)out_dev);
}

extern "C" int ifs_far_field(ifs_ctx *c, const double *x, int64_t n, int32_t ndir, const double *theta,
                             const double *phi, double *out) {
    if (!c || !x || !theta || !phi || !out || n != ifs_vector_length(c) || ndir < 0) return IFS_E_ARG;
    if (ndir == 0) return IFS_OK;
    // one allocation: x, theta, phi, out, tables and parts
    const int64_t entries = (int64_t)ndir * c->N * (c->N + 2);
    const int parts = ifs::ff_parts(c->N, ndir, INT64_MAX);
    ifs::DevBuf d;
    int rc;
    if ((rc = d.alloc(16ull * (n + 3ll * ndir + entries + 2ll * ndir * (parts > 1 ? parts : 0))))) return rc;
    double2 *dx = d.as<double2>(), *dout = dx + n;
    double *dt = (double *)(dout + 2ll * ndir), *dph = dt + ndir;
    hipStream_t s = c->stream;
    if (hipMemcpyAsync(dx, x, 16ull * n, hipMemcpyHostToDevice, s) != hipSuccess ||
        hipMemcpyAsync(dt, theta, 8ull * ndir, hipMemcpyHostToDevice, s) != hipSuccess ||
        hipMemcpyAsync(dph, phi, 8ull * ndir, hipMemcpyHostToDevice, s) != hipSuccess ||
        (rc = ifs::ff_launch(c, dx, ndir, dt, dph, dout + 3ll * ndir, parts, dout)) ||
        hipMemcpyAsync(out, dout, 32ull * ndir, hipMemcpyDeviceToHost, s) != hipSuccess)
        rc = rc ? rc : IFS_E_HIP;
    return hipStreamSynchronize(s) == hipSuccess ? rc : IFS_E_HIP;
}

extern "C" int ifs_amplitude_matrix(int32_t ndir, const double *phi, const double *Fx, const double *Fy, double *S) {
    if (ndir < 0 || !phi || !Fx || !Fy || !S) return IFS_E_ARG;
    const cplx I(0.0, 1.0);
    const cplx *fx = (const cplx *)Fx, *fy = (const cplx *)Fy;
    cplx *s = (cplx *)S;
    for (int i = 0; i < ndir; ++i) {
        double c = std::cos(phi[i]), sn = std::sin(phi[i]);
        cplx xt = fx[2 * i], xp = fx[2 * i + 1], yt = fy[2 * i], yp = fy[2 * i + 1];
        s[4 * i + 0] = I * (xp * sn - yp * c);         // S1
        s[4 * i + 1] = -I * (xt * c + yt * sn);        // S2
        s[4 * i + 2] = -I * (xt * sn - yt * c);        // S3
        s[4 * i + 3] = I * (xp * c + yp * sn);         // S4
    }
    return IFS_OK;
}

extern "C" int ifs_mueller(int32_t ndir, const double *S, double *M) {
    if (ndir < 0 || !S || !M) return IFS_E_ARG;
    const cplx *s = (const cplx *)S;
    for (int i = 0; i < ndir; ++i) {
        cplx S1 = s[4 * i], S2 = s[4 * i + 1], S3 = s[4 * i + 2], S4 = s[4 * i + 3];
        double a1 = std::norm(S1), a2 = std::norm(S2), a3 = std::norm(S3), a4 = std::norm(S4);
        double *m = M + 16 * i;
        m[0] = 0.5 * (a2 + a3 + a4 + a1);
        m[1] = 0.5 * (a2 - a3 + a4 - a1);
        m[2] = std::real(S2 * std::conj(S3) + S1 * std::conj(S4));
        m[3] = std::imag(S2 * std::conj(S3) - S1 * std::conj(S4));
        m[4] = 0.5 * (a2 - a4 + a3 - a1);
        m[5] = 0.5 * (a2 - a3 - a4 + a1);
        m[6] = std::real(S2 * std::conj(S3) - S1 * std::conj(S4));
        m[7] = std::imag(S2 * std::conj(S3) + S1 * std::conj(S4));
        m[8] = std::real(S2 * std::conj(S4) + S1 * std::conj(S3));
        m[9] = std::real(S2 * std::conj(S4) - S1 * std::conj(S3));
        m[10] = std::real(S1 * std::conj(S2) + S3 * std::conj(S4));
        m[11] = std::imag(S2 * std::conj(S1) + S4 * std::conj(S3));
        m[12] = std::imag(S4 * std::conj(S2) + S1 * std::conj(S3));
        m[13] = std::imag(S4 * std::conj(S2) - S1 * std::conj(S3));
        m[14] = std::imag(S1 * std::conj(S2) - S3 * std::conj(S4));
        m[15] = std::real(S1 * std::conj(S2) - S3 * std::conj(S4));
    }
    return IFS_OK;
}
