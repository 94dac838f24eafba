// Sphere <-> leaf box translations (P2M, L2P) through samples of the box's field (gfx950).
//
// In the helicity basis a regular translation by d is the factor e^{i k s . d} on the plane
// waves s (see ifs_pw.hip).  P2M: every sphere of a box is sampled on the box's grid, times
// its factor, and added up; one analysis per box gives the multipole coefficients.  L2P: one
// synthesis per box, then every sphere projects the samples times its factor.  The grid
// integrates degree L + N + k r + 8 (k r)^{1/3} + 30, about half the rows and azimuths that the
// box translations need.  A sphere of order N costs about (8 N + 150) flops per sample of a
// quarter circle: the four azimuths phi + j pi/2 share their sums over m (m mod 4) and two
// sine-cosine pairs.  The one-by-one translations read a Wigner table of 16 K L^2 bytes per
// sphere and product.  P2M + L2P against them: 2500 spheres, 512 boxes of order 97 10.1 -> 4.7
// ms; 333 droplets, 64 boxes of order 410 13.5 -> 8.0 ms; 700 spheres with four right-hand
// sides 16.8 -> 6.8 ms; first products of a new cluster 79 -> 45 ms and 151 -> 79 ms.
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>

#include "ifs_leaf.h"

namespace ifs {

namespace {
__device__ __forceinline__ double2 cm(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
}  // namespace

// us[position][n (n+1)/2 + m] = sqrt((2n+1)/2) d^n_{m,1}, n = 1..Nmax, 0 <= m <= n: thread per
// (position, m); position t < Q2 is node t, t >= Q2 its mirror.
__global__ void k_leaf_utable(int Nmax, int Q2, int ucols, const double *__restrict__ mu, double *__restrict__ us) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int m = blockIdx.y;
    if (t >= 2 * Q2) return;
    const double x = t < Q2 ? mu[t] : -mu[t - Q2];
    const double ch = sqrt(0.5 * (1.0 + x)), sh = sqrt(0.5 * (1.0 - x));
    double d1, d2 = 0.0, sp = 0.0;
    if (m == 0) {
        d1 = sqrt(2.0) * ch * sh;
    } else {
        double c = 1.0, p = 1.0;  // d^m_{m,1} = sqrt((2m)!/((m+1)!(m-1)!)) ch^{m+1} (-sh)^{m-1}
        for (int i = 2; i <= m; ++i) {
            c *= (double)(2 * i) * (double)(2 * i - 1) / (4.0 * (double)(i + 1) * (double)(i - 1));
            p *= -2.0 * ch * sh;
        }
        d1 = sqrt(c) * p * ch * ch;
    }
    double *o = us + (int64_t)t * ucols + m;
    const int n0 = m < 1 ? 1 : m;
    const double mm = (double)m * m;
    for (int n = n0; n <= Nmax; ++n) {
        if (n > n0) {
            const double nn = n, n1 = nn - 1.0;
            const double sc = sqrt((nn * nn - mm) * (nn * nn - 1.0));
            const double d = ((2.0 * nn - 1.0) * (nn * n1 * x - (double)m) * d1 - nn * sp * d2) / (n1 * sc);
            d2 = d1;
            d1 = d;
            sp = sc;
        }
        o[n * (n + 1) / 2] = sqrt(n + 0.5) * d1;
    }
}

// Coefficient of degree n in the row sum of (helicity, m) at a position, from the table rows of
// the position and of its mirror: U_{n,m}^- = (-1)^{n+m} U_{n,m}^+ (mirror), U_{n,-m}^+- = (-1)^{m+1} U_{n,m}^-+.
struct URow {
    const double *u;
    double s0, sn;  // sign at n even, n odd
    __device__ __forceinline__ URow(const double *row, const double *mir, int hel, int m) {
        const int am = m < 0 ? -m : m;
        const bool mirror = (hel == 1) != (m < 0);
        const double sm = (am & 1) ? -1.0 : 1.0;
        u = (mirror ? mir : row) + am;
        s0 = (mirror ? sm : 1.0) * (m < 0 ? -sm : 1.0);
        sn = mirror ? -s0 : s0;
    }
    __device__ __forceinline__ double at(int n) const { return ((n & 1) ? sn : s0) * u[n * (n + 1) / 2]; }
};

// Row sums of the spheres, g[(sphere - s0)][rhs][position][helicity][m + Nmax] = sum_n U x: block
// (sphere, eight rows), thread per (helicity, m).
constexpr int LROWS = 8;
__global__ __launch_bounds__(128) void k_leaf_rows(LeafArg a, const LeafSphere *__restrict__ sph, int s0,
                                                   const double2 *__restrict__ xh, int64_t ldx,
                                                   double2 *__restrict__ g) {
    const int nrhs = a.p.nbr / a.nb;
    const int si = blockIdx.x / nrhs, rhs = blockIdx.x % nrhs;
    const LeafSphere S = sph[s0 + si];
    const int M = 2 * S.N + 1, W = 2 * a.Nmax + 1, R2 = a.p.R2;
    const double2 *xa = xh + rhs * ldx + S.off, *xb = xa + (int64_t)S.N * (S.N + 2);
    double2 *go = g + ((int64_t)si * nrhs + rhs) * 2 * a.p.Q2 * 2 * W;
    for (int o = threadIdx.x; o < 2 * M; o += 128) {
        const int h = o >= M, m = o - h * M - S.N;
        const int am = m < 0 ? -m : m;
        const bool mirror = (h == 1) != (m < 0);
        const double sm = (am & 1) ? -1.0 : 1.0;
        const double se = (mirror ? sm : 1.0) * (m < 0 ? -sm : 1.0), so = mirror ? -se : se;
        const double *u[LROWS];
        double re[LROWS], im[LROWS];
#pragma unroll
        for (int r = 0; r < LROWS; ++r) {
            const int lr = min((int)blockIdx.y * LROWS + r, 2 * R2 - 1);
            const bool north = (lr < R2) != mirror;
            u[r] = a.us + (int64_t)(a.p.j0 + (lr < R2 ? lr : lr - R2) + (north ? 0 : a.p.Q2)) * a.ucols + am;
            re[r] = im[r] = 0.0;
        }
        for (int n = am < 1 ? 1 : am; n <= S.N; ++n) {
            const double2 p = xa[n * n - 1 + n + m], q = xb[n * n - 1 + n + m];
            const double sg = (n & 1) ? so : se;
            const double xr = sg * (h ? p.x - q.x : p.x + q.x), xi = sg * (h ? p.y - q.y : p.y + q.y);
            const int e = n * (n + 1) / 2;
#pragma unroll
            for (int r = 0; r < LROWS; ++r) {
                const double w = u[r][e];
                re[r] = fma(w, xr, re[r]);
                im[r] = fma(w, xi, im[r]);
            }
        }
#pragma unroll
        for (int r = 0; r < LROWS; ++r) {
            const int lr = blockIdx.y * LROWS + r;
            if (lr >= 2 * R2) break;
            const int pos = a.p.j0 + (lr < R2 ? lr : lr - R2 + a.p.Q2);
            go[(int64_t)(2 * pos + h) * W + m + a.Nmax] = make_double2(re[r], im[r]);
        }
    }
}

// P2M samples: block (box, row, tile of quarter azimuths), spheres one after another: a thread
// adds its four azimuths; the next sphere's row sums come into the other half of LDS meanwhile.
__global__ __launch_bounds__(64, 3) void k_leaf_p2m(LeafArg a, const LeafSphere *__restrict__ sph,
                                                  const int32_t *__restrict__ first, int s0, int s1,
                                                  const double2 *__restrict__ grow, int accumulate) {
    extern __shared__ double2 gs[];  // [2][2][2 Nmax + 1]
    const int box = blockIdx.x, lr = blockIdx.y;
    const int nrhs = a.p.nbr / a.nb;
    const int tiles = gridDim.z / nrhs;
    const int at = blockIdx.z % tiles, rhs = blockIdx.z / tiles;
    const int R2 = a.p.R2;
    const int node = a.p.j0 + (lr < R2 ? lr : lr - R2);
    const int N = a.p.N[node], N4 = N >> 2;
    if (at * 64 >= N4) return;
    const int W = 2 * a.Nmax + 1;
    const int pos = lr < R2 ? node : a.p.Q2 + node;
    const double mu = a.mu[node], z = lr < R2 ? mu : -mu, st = sqrt((1.0 - mu) * (1.0 + mu));
    const int i = at * 64 + threadIdx.x;
    const bool on = i < N4;
    double sn, cs;
    sincospi(2.0 * (double)i / (double)N, &sn, &cs);
    const double2 e1 = make_double2(cs, sn), e2 = cm(e1, e1), e4 = cm(e2, e2);
    double2 acc[2][4];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[h][j] = make_double2(0.0, 0.0);
    const int qb = max(first[box], s0), qe = min(first[box + 1], s1);
    auto stage = [&](int q) {
        const int M = 2 * sph[q].N + 1;
        const double2 *src = grow + (((int64_t)(q - s0) * nrhs + rhs) * 2 * a.p.Q2 + pos) * 2 * W + a.Nmax - sph[q].N;
        double2 *dst = gs + ((q - qb) & 1) * 2 * W;
        for (int o = threadIdx.x; o < 2 * M; o += 64) dst[o] = src[o < M ? o : o - M + W];
    };
    if (qb < qe) stage(qb);
    for (int q = qb; q < qe; ++q) {
        const LeafSphere S = sph[q];
        const int M = 2 * S.N + 1;
        const double2 *g = gs + ((q - qb) & 1) * 2 * W;
        __syncthreads();
        if (q + 1 < qe) stage(q + 1);
        if (!on) continue;
        // factors at the four azimuths: e^{i (z v_z +- A)}, e^{i (z v_z +- B)}
        double s0, c0, s1, c1, s2, c2;
        sincos(z * S.v[2], &s0, &c0);
        sincos(st * (cs * S.v[0] + sn * S.v[1]), &s1, &c1);
        sincos(st * (-sn * S.v[0] + cs * S.v[1]), &s2, &c2);
        const double2 w0 = make_double2(c0, s0);
        const double2 f[4] = {cm(w0, make_double2(c1, s1)), cm(w0, make_double2(c2, s2)),
                              cm(w0, make_double2(c1, -s1)), cm(w0, make_double2(c2, -s2))};
        // m = o - B, o = 0 .. B + N with B = N rounded up to 4: the class of m mod 4 is o mod 4;
        // each class by Horner in e^{4 i phi}
        const int B = (S.N + 3) & ~3, lo = B - S.N;
        double sB, cB;
        sincospi(-2.0 * (double)((B * i) % N) / (double)N, &sB, &cB);
        const double2 eB = make_double2(cB, sB);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const double2 *G = g + h * M;
            double2 t[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) t[c] = make_double2(0.0, 0.0);
            for (int k = (B + S.N) >> 2; k >= 0; --k)
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int o = 4 * k + c - lo;
                    const double2 v = o >= 0 && o < M ? G[o] : make_double2(0.0, 0.0);
                    t[c] = make_double2(fma(t[c].x, e4.x, fma(-t[c].y, e4.y, v.x)),
                                        fma(t[c].x, e4.y, fma(t[c].y, e4.x, v.y)));
                }
            t[0] = cm(eB, t[0]);
            t[1] = cm(eB, cm(e1, t[1]));
            t[2] = cm(eB, cm(e2, t[2]));
            t[3] = cm(eB, cm(cm(e1, e2), t[3]));
            // azimuth phi + j pi/2: the classes times i^{j c}
            const double2 p = make_double2(t[0].x + t[2].x, t[0].y + t[2].y), r = make_double2(t[0].x - t[2].x, t[0].y - t[2].y);
            const double2 u = make_double2(t[1].x + t[3].x, t[1].y + t[3].y);
            const double2 v = make_double2(-(t[1].y - t[3].y), t[1].x - t[3].x);  // i (t1 - t3)
            const double2 F[4] = {make_double2(p.x + u.x, p.y + u.y), make_double2(r.x + v.x, r.y + v.y),
                                  make_double2(p.x - u.x, p.y - u.y), make_double2(r.x - v.x, r.y - v.y)};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const double2 y = cm(f[j], F[j]);
                acc[h][j].x += y.x;
                acc[h][j].y += y.y;
            }
        }
    }
    if (!on) return;
    const double w = a.mu[a.p.Q2 + node] / (double)N;
    double2 *o = a.p.H + 2 * a.p.cpre[lr] * a.p.nbr + (int64_t)(rhs * a.nb + box) * N + i;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            double2 *d = o + (int64_t)h * a.p.nbr * N + j * N4;
            double2 v = make_double2(w * acc[h][j].x, w * acc[h][j].y);
            if (accumulate) {
                v.x += d->x;
                v.y += d->y;
            }
            *d = v;
        }
}

// L2P, one row of one sphere per block: samples times the factor, reduced to the four classes of
// m mod 4 per quarter azimuth in LDS, then a thread per (helicity, m, part of the azimuths).
__global__ __launch_bounds__(128) void k_leaf_l2p(LeafArg a, const LeafSphere *__restrict__ sph, int s0, int N4max,
                                                  double2 *__restrict__ gout) {
    extern __shared__ double2 sm[];  // [2][4][N4max], then partial sums [2][2 Nmax + 1][parts]
    const int nrhs = a.p.nbr / a.nb;
    const int si = blockIdx.x / nrhs, rhs = blockIdx.x % nrhs;
    const int lr = blockIdx.y;
    const LeafSphere S = sph[s0 + si];
    const int R2 = a.p.R2;
    const int node = a.p.j0 + (lr < R2 ? lr : lr - R2);
    const int N = a.p.N[node], N4 = N >> 2;
    const int pos = lr < R2 ? node : a.p.Q2 + node;
    const double mu = a.mu[node], z = lr < R2 ? mu : -mu, st = sqrt((1.0 - mu) * (1.0 + mu));
    const double wt = a.mu[a.p.Q2 + node] / (double)N;
    double s0_, c0_;
    sincos(z * S.v[2], &s0_, &c0_);
    const double2 w0 = make_double2(wt * c0_, wt * s0_);
    const double2 *F = a.p.F + 2 * a.p.cpre[lr] * a.p.nbr + (int64_t)(rhs * a.nb + S.box) * N;
    for (int i = threadIdx.x; i < N4; i += 128) {
        double sn, cs, s1, c1, s2, c2;
        sincospi(2.0 * (double)i / (double)N, &sn, &cs);
        sincos(st * (cs * S.v[0] + sn * S.v[1]), &s1, &c1);
        sincos(st * (-sn * S.v[0] + cs * S.v[1]), &s2, &c2);
        const double2 f[4] = {cm(w0, make_double2(c1, s1)), cm(w0, make_double2(c2, s2)),
                              cm(w0, make_double2(c1, -s1)), cm(w0, make_double2(c2, -s2))};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            double2 p[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) p[j] = cm(f[j], F[(int64_t)h * a.p.nbr * N + j * N4 + i]);
            // class c: sum_j i^{-j c} p_j
            const double2 e = make_double2(p[0].x + p[2].x, p[0].y + p[2].y), d = make_double2(p[0].x - p[2].x, p[0].y - p[2].y);
            const double2 u = make_double2(p[1].x + p[3].x, p[1].y + p[3].y);
            const double2 v = make_double2(p[1].y - p[3].y, -(p[1].x - p[3].x));  // -i (p1 - p3)
            double2 *o = sm + h * 4 * N4max + i;
            o[0] = make_double2(e.x + u.x, e.y + u.y);
            o[N4max] = make_double2(d.x + v.x, d.y + v.y);
            o[2 * N4max] = make_double2(e.x - u.x, e.y - u.y);
            o[3 * N4max] = make_double2(d.x - v.x, d.y - v.y);
        }
    }
    __syncthreads();
    const int M = 2 * S.N + 1, M2 = 2 * M;
    double2 *go = gout + (((int64_t)si * nrhs + rhs) * 2 * a.p.Q2 + pos) * 2 * (2 * a.Nmax + 1);
    const int parts = M2 <= 128 ? 128 / M2 : 1;
    double2 *red = sm + 8 * N4max;
    for (int o0 = 0; o0 < M2; o0 += 128) {
        const int id = o0 + threadIdx.x;
        const int o = parts > 1 ? threadIdx.x % M2 : id, part = parts > 1 ? threadIdx.x / M2 : 0;
        if (o < M2 && part < parts) {
            const int h = o >= M, m = o - h * M - S.N;
            const int b = N4 * part / parts, e = N4 * (part + 1) / parts;
            const double2 *x = sm + (h * 4 + (m & 3)) * N4max;
            double ss, cc, sr, cr;
            sincospi(-2.0 * (double)m / (double)N, &sr, &cr);
            double re = 0.0, im = 0.0;
            for (int i0 = b; i0 < e; i0 += 32) {  // the turning factor afresh every 32 azimuths
                const int mi = (int)(((int64_t)m * i0) % N);
                sincospi(-2.0 * (double)mi / (double)N, &ss, &cc);
                const int ie = min(e, i0 + 32);
                for (int i = i0; i < ie; ++i) {
                    const double2 v = x[i];
                    re = fma(v.x, cc, fma(-v.y, ss, re));
                    im = fma(v.x, ss, fma(v.y, cc, im));
                    const double t = cc * cr - ss * sr;
                    ss = fma(cc, sr, ss * cr);
                    cc = t;
                }
            }
            if (parts > 1)
                red[part * M2 + o] = make_double2(re, im);
            else
                go[h * (2 * a.Nmax + 1) + m + a.Nmax] = make_double2(re, im);
        }
    }
    if (parts > 1) {
        __syncthreads();
        for (int o = threadIdx.x; o < M2; o += 128) {
            double2 t = red[o];
            for (int p = 1; p < parts; ++p) {
                t.x += red[p * M2 + o].x;
                t.y += red[p * M2 + o].y;
            }
            const int h = o >= M, m = o - h * M - S.N;
            go[h * (2 * a.Nmax + 1) + m + a.Nmax] = t;
        }
    }
}

// acc(n, m) += sum over the positions of U g: thread per entry, block per (sphere, entries).
__global__ __launch_bounds__(256) void k_leaf_sum(LeafArg a, const LeafSphere *__restrict__ sph, int s0, int nrhs,
                                                  const double2 *__restrict__ gin, double2 *__restrict__ acc,
                                                  int64_t ldacc) {
    __shared__ double2 red[2][4][64];
    const int si = blockIdx.x / nrhs, rhs = blockIdx.x % nrhs;
    const LeafSphere S = sph[s0 + si];
    const int nent = S.N * (S.N + 2);
    if ((int)blockIdx.y * 64 >= nent) return;
    const int e = blockIdx.y * 64 + (threadIdx.x & 63), w = threadIdx.x >> 6;
    const int W = 2 * a.Nmax + 1, Q = 2 * a.p.Q2;
    double2 t[2] = {make_double2(0.0, 0.0), make_double2(0.0, 0.0)};
    if (e < nent) {
        int n = (int)sqrt((double)(e + 1));
        while ((n + 1) * (n + 1) - 1 <= e) ++n;
        while (n * n - 1 > e) --n;
        const int m = e - (n * n - 1) - n;
        const double2 *g = gin + ((int64_t)si * nrhs + rhs) * Q * 2 * W + m + a.Nmax;
        for (int p = w; p < Q; p += 4) {  // a quarter of the positions per wave
            const int mp = p < a.p.Q2 ? p + a.p.Q2 : p - a.p.Q2;
            const double *row = a.us + (int64_t)p * a.ucols, *mir = a.us + (int64_t)mp * a.ucols;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const URow U(row, mir, h, m);
                const double u = U.at(n);
                const double2 v = g[(int64_t)(2 * p + h) * W];
                t[h].x = fma(u, v.x, t[h].x);
                t[h].y = fma(u, v.y, t[h].y);
            }
        }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) red[h][w][threadIdx.x & 63] = t[h];
    __syncthreads();
    if (w != 0 || e >= nent) return;
    double2 s[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        s[h] = red[h][0][threadIdx.x];
#pragma unroll
        for (int q = 1; q < 4; ++q) {
            s[h].x += red[h][q][threadIdx.x].x;
            s[h].y += red[h][q][threadIdx.x].y;
        }
    }
    double2 *d = acc + rhs * ldacc + S.off + e;
    d[0] = make_double2(d[0].x + 0.5 * (s[0].x + s[1].x), d[0].y + 0.5 * (s[0].y + s[1].y));
    d[nent] = make_double2(d[nent].x + 0.5 * (s[0].x - s[1].x), d[nent].y + 0.5 * (s[0].y - s[1].y));
}

void launch_leaf_utable(int Nmax, int Q2, int ucols, const double *mu, double *us, hipStream_t s) {
    hipLaunchKernelGGL(k_leaf_utable, dim3((2 * Q2 + 63) / 64, Nmax + 1), dim3(64), 0, s, Nmax, Q2, ucols, mu, us);
}
void launch_leaf_p2m(const LeafArg &a, const LeafSphere *sph, const int32_t *first, int s0, int ns, const double2 *xh,
                     int64_t ldx, int nrhs, int maxN, double2 *g, int accumulate, hipStream_t s) {
    if (ns > 0)
        hipLaunchKernelGGL(k_leaf_rows, dim3(ns * nrhs, (2 * a.p.R2 + LROWS - 1) / LROWS), dim3(128), 0, s, a, sph, s0,
                           xh, ldx, g);
    const int tiles = (maxN / 4 + 63) / 64;
    hipLaunchKernelGGL(k_leaf_p2m, dim3(a.nb, 2 * a.p.R2, tiles * nrhs), dim3(64),
                       leaf_p2m_lds(a.Nmax), s, a, sph, first, s0, s0 + ns, g, accumulate);
}
void launch_leaf_l2p(const LeafArg &a, const LeafSphere *sph, int s0, int ns, int nrhs, int maxN, double2 *g,
                     hipStream_t s) {
    if (ns <= 0) return;
    const int n4 = maxN / 4;
    hipLaunchKernelGGL(k_leaf_l2p, dim3(ns * nrhs, 2 * a.p.R2), dim3(128), leaf_l2p_lds(maxN), s,
                       a, sph, s0, n4, g);
}
void launch_leaf_sum(const LeafArg &a, const LeafSphere *sph, int s0, int ns, int nrhs, const double2 *g, double2 *acc,
                     int64_t ldacc, hipStream_t s) {
    if (ns <= 0) return;
    hipLaunchKernelGGL(k_leaf_sum, dim3(ns * nrhs, (a.Nmax * (a.Nmax + 2) + 63) / 64), dim3(256), 0, s, a, sph, s0,
                       nrhs, g, acc, ldacc);
}

}  // namespace ifs
