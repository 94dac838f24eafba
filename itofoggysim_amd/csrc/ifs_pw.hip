// Box-to-box translations (M2L) of one octree level in the plane-wave basis (gfx950).
//
// In the helicity basis x_+- = x_a +- x_b every outgoing -> regular translation is
//   D_nm = sum_{nu,mu} int U_n^m(mu) U_nu^mu(mu) e^{i(mu-m)phi} T(s . d) ds/2pi C_{nu mu},
//   U_n^m = sqrt((2n+1)/2) d^n_{m,+-1},  T(x) = sum_{p <= 2L} i^p (2p+1) h1_p(t) P_p(x),
// exactly (the quadrature below integrates every degree up to 4L): with samples
// F(theta, phi) of a box's field on one grid, a translation is a product by T per sample.
// A box costs one synthesis and one analysis (32 L^3 flops) instead of about 21 L^3 per
// translation, of which it has a hundred; a translation costs about 8 L^2 samples.
//
// Rows theta: Gauss-Legendre nodes in mirrored pairs (position t and t + Q2), so one
// table U of helicity +1 serves both: U^-_n,m(theta) = (-1)^{n+m} U^+_n,m(pi - theta) and
// U_{n,-m}^+- = (-1)^{m+1} U_{n,m}^-+.  Azimuths per row: N >= 2 mF + mT + 1 with mF and mT the largest
// orders of the field and of T that reach 1e-16 there (U falls like a Bessel function
// J_m(n sin(theta)) beyond m = n sin(theta)).
//
// Launches per chunk of rows: GEMM (X -> G, orders x rows x boxes), FFT along the
// azimuth in LDS (G -> F), products (F -> H), FFT back (H -> G), GEMM (G -> Xd).
//
// Bound by the products' reads of T and of samples (16 bytes of T per 16 flops, 16 TB/s from
// L2) and by the transforms' passes over G and F.  M2L against class products of rotations and shifts:
// 64 boxes of order 410 (3004 translations) 120 -> 16.5 ms, 512 + 64 boxes of orders 97
// and 174 (56046) 64 -> 17 ms, orders 45 and 77 (56448) 13.7 -> 5.7 ms (with what the class
// products keep of near offsets).  Against the direct product of 200 / 600 spheres the
// MLFMM is off by 4.4e-14 / 1.0e-13 (class products 3.7e-10 / 5.7e-9).
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>

#include "ifs_pw.h"

namespace ifs {

namespace {
typedef double dv4 __attribute__((ext_vector_type(4)));
// Blocks that follow one another share cache lines: the 8 dies take blocks in turn, so
// give each die a run of consecutive work.
__device__ __forceinline__ int64_t die_order(int64_t b, int64_t n) {
    const int64_t per = n >> 3;
    return b < per * 8 ? (b & 7) * per + (b >> 3) : b;
}
}  // namespace

// U[(ucnt(m) + n - n0) ustr + pos]: block (rows, m), thread per row.
__global__ void k_pw_utable(int L, int Q2, int j0, int R2, int a0, int a1, int64_t ustr, const double *__restrict__ mu,
                            double *__restrict__ U) {
    const int lr = blockIdx.x * blockDim.x + threadIdx.x;
    const int m = blockIdx.y;
    if (lr >= 2 * R2) return;
    const bool south = lr >= R2;
    const int j = j0 + (south ? lr - R2 : lr);
    const double x = south ? -mu[j] : mu[j];
    double *o = U + pw_ucnt(m, L) * ustr + (south ? a1 + lr - R2 : a0 + lr);
    const double ch = sqrt(0.5 * (1.0 + x)), sh = sqrt(0.5 * (1.0 - x));
    double d1;
    if (m == 0) {
        d1 = sqrt(2.0) * ch * sh;
    } else {
        // d^m_{m,1} = sqrt((2m)!/((m+1)!(m-1)!)) ch^{m+1} (-sh)^{m-1}
        double c = 1.0, p = 1.0;
        const double s = -2.0 * ch * sh;
        for (int i = 2; i <= m; ++i) {
            c *= (double)(2 * i) * (double)(2 * i - 1) / (4.0 * (double)(i + 1) * (double)(i - 1));
            p *= s;
        }
        d1 = sqrt(c) * p * ch * ch;
    }
    double d2 = 0.0;
    const int n0 = m < 1 ? 1 : m;
    const double mm = (double)m * m;
    double sp = 0.0;  // sqrt(((n-1)^2 - m^2)((n-1)^2 - 1))
    for (int n = n0; n <= L; ++n) {
        if (n > n0) {
            const double nn = n, n1 = nn - 1.0;
            const double sc = sqrt((nn * nn - mm) * (nn * nn - 1.0));
            const double d = ((2.0 * nn - 1.0) * (nn * n1 * x - (double)m) * d1 - nn * sp * d2) / (n1 * sc);
            d2 = d1;
            d1 = d;
            sp = sc;
        }
        *o = sqrt(n + 0.5) * d1;
        o += ustr;
    }
}

// c_p = i^p (2p+1) h1_p(t), p = 0..P: one thread per table (j downward, y upward).
__global__ void k_pw_hankel(int P, const double *__restrict__ t, const int32_t *__restrict__ terms,
                            double2 *__restrict__ hh) {
    if (threadIdx.x != 0) return;
    const double x = t[blockIdx.x];
    double2 *h = hh + (int64_t)blockIdx.x * (P + 1);
    const double big = (double)P > x ? (double)P : x;
    const int nstart = (int)big + 30 + (int)sqrt(40.0 * big);
    double fp1 = 0.0, f = 1e-200;
    for (int n = nstart; n >= 1; --n) {
        const double fm1 = (2.0 * n + 1.0) / x * f - fp1;
        fp1 = f;
        f = fm1;
        if (n - 1 <= P) h[n - 1].x = f;
        if (fabs(f) > 1e200) {
            f *= 1e-200;
            fp1 *= 1e-200;
            for (int q = n - 1; q <= P; ++q) h[q].x *= 1e-200;
        }
    }
    double sx, cx;
    sincos(x, &sx, &cx);
    const double j0 = sx / x, j1 = sx / (x * x) - cx / x;
    const double scale = fabs(j1) > fabs(j0) ? j1 / h[1].x : j0 / h[0].x;
    double ym1 = -cx / x, y = -cx / (x * x) - sx / x;
    for (int p = 0; p <= P; ++p) {
        const double jr = h[p].x * scale, yr = ym1, c = p > terms[blockIdx.x] ? 0.0 : 2.0 * p + 1.0;
        switch (p & 3) {
            case 0: h[p] = make_double2(c * jr, c * yr); break;
            case 1: h[p] = make_double2(-c * yr, c * jr); break;
            case 2: h[p] = make_double2(-c * jr, -c * yr); break;
            default: h[p] = make_double2(c * yr, -c * jr);
        }
        const double yn = (2.0 * p + 3.0) / x * y - ym1;
        ym1 = y;
        y = yn;
    }
}

// T of a canonical offset at the rows' nodes, times w_q / N.  Legendre polynomials by
// differences in 1 - |x| (exact where x rounds to 1).  Block (azimuths, row, table).
__global__ __launch_bounds__(256) void k_pw_ttable(int P, int Q2, int j0, int R2, int a0, int a1,
                                                   const double *__restrict__ mu, const double *__restrict__ canon,
                                                   const int32_t *__restrict__ N, const int64_t *__restrict__ tpre,
                                                   int64_t tsn, const double2 *__restrict__ hh,
                                                   double2 *__restrict__ T, float2 *__restrict__ T32) {
    extern __shared__ double2 h[];
    const int lr = blockIdx.y, c = blockIdx.z;
    const bool south = lr >= R2;
    const int j = j0 + (south ? lr - R2 : lr);
    const int n = N[j];
    if ((int)(blockIdx.x * blockDim.x) >= n) return;
    for (int p = threadIdx.x; p <= P; p += blockDim.x) h[p] = hh[(int64_t)c * (P + 1) + p];
    __syncthreads();
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double z = south ? -mu[j] : mu[j], st = sqrt((1.0 - mu[j]) * (1.0 + mu[j]));
    double sn, cs;
    sincospi(2.0 * (double)i / (double)n, &sn, &cs);
    const double *d = canon + 4 * c;
    const double vx = st * cs, vy = st * sn;
    const double x = vx * d[0] + vy * d[1] + z * d[2];
    const double sg = x < 0.0 ? -1.0 : 1.0;
    const double ex = vx - sg * d[0], ey = vy - sg * d[1], ez = z - sg * d[2];
    const double dl = 0.5 * (ex * ex + ey * ey + ez * ez);  // 1 - |x|
    double pc = 1.0, df = 0.0, ar = 0.0, ai = 0.0, f = 1.0;
    for (int p = 0; p <= P; ++p) {
        const double2 v = h[p];
        const double q = f * pc;
        ar = fma(q, v.x, ar);
        ai = fma(q, v.y, ai);
        const double dp = p;
        df = (dp * df - (2.0 * dp + 1.0) * dl * pc) / (dp + 1.0);
        pc += df;
        f *= sg;
    }
    const double w = mu[Q2 + j] / (double)n;
    const int pos = south ? a1 + lr - R2 : a0 + lr;
    const int64_t o = (int64_t)c * tsn + tpre[pos] + i;
    if (T32)
        T32[o] = make_float2((float)(w * ar), (float)(w * ai));
    else
        T[o] = make_double2(w * ar, w * ai);
}

// Pool -> X[order][helicity][degree][box]: 16 entries x 32 boxes through LDS.
__global__ __launch_bounds__(256) void k_pw_pack(PwArg a, int nb, int64_t off, const double2 *__restrict__ C,
                                                 int64_t stride) {
    __shared__ double2 s[2][16][33];
    const int nent = a.L * (a.L + 2);
    const int e0 = blockIdx.x * 16, b0 = blockIdx.y * 32;
    for (int i = threadIdx.x; i < 512; i += 256) {
        const int e = e0 + (i & 15), b = b0 + (i >> 4);
        if (e < nent && b < a.nbr) {
            const double2 *p = C + (int64_t)(b / nb) * stride + off + (int64_t)(b % nb) * 2 * nent + e;
            const double2 u = p[0], v = p[nent];
            s[0][i & 15][i >> 4] = make_double2(u.x + v.x, u.y + v.y);
            s[1][i & 15][i >> 4] = make_double2(u.x - v.x, u.y - v.y);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 512; i += 256) {
        const int e = e0 + (i >> 5), b = b0 + (i & 31);
        if (e >= nent || b >= a.nbr) continue;
        int n = (int)sqrt((double)(e + 1));
        while ((n + 1) * (n + 1) - 1 <= e) ++n;
        while (n * n - 1 > e) --n;
        const int m = e - (n * n - 1) - n;
        const int am = m < 0 ? -m : m;
        const int64_t row = 2 * pw_xcnt(m, a.L) + n - (am < 1 ? 1 : am);
        a.X[row * a.nbr + b] = s[0][i >> 5][i & 31];
        a.X[(row + pw_cn(m, a.L)) * a.nbr + b] = s[1][i >> 5][i & 31];
    }
}

// D += the analysed expansions.
__global__ __launch_bounds__(256) void k_pw_unpack(PwArg a, int nb, int64_t off, double2 *__restrict__ D,
                                                   int64_t stride) {
    __shared__ double2 s[2][16][33];
    const int nent = a.L * (a.L + 2);
    const int e0 = blockIdx.x * 16, b0 = blockIdx.y * 32;
    for (int i = threadIdx.x; i < 512; i += 256) {
        const int e = e0 + (i >> 5), b = b0 + (i & 31);
        if (e >= nent || b >= a.nbr) continue;
        int n = (int)sqrt((double)(e + 1));
        while ((n + 1) * (n + 1) - 1 <= e) ++n;
        while (n * n - 1 > e) --n;
        const int m = e - (n * n - 1) - n;
        const int am = m < 0 ? -m : m;
        const int64_t row = 2 * pw_xcnt(m, a.L) + n - (am < 1 ? 1 : am);
        const double2 u = a.Xd[row * a.nbr + b], v = a.Xd[(row + pw_cn(m, a.L)) * a.nbr + b];
        s[0][i >> 5][i & 31] = make_double2(0.5 * (u.x + v.x), 0.5 * (u.y + v.y));
        s[1][i >> 5][i & 31] = make_double2(0.5 * (u.x - v.x), 0.5 * (u.y - v.y));
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 512; i += 256) {
        const int e = e0 + (i & 15), b = b0 + (i >> 4);
        if (e >= nent || b >= a.nbr) continue;
        double2 *p = D + (int64_t)(b / nb) * stride + off + (int64_t)(b % nb) * 2 * nent + e;
        const double2 u = s[0][i & 15][i >> 4], v = s[1][i & 15][i >> 4];
        p[0] = make_double2(p[0].x + u.x, p[0].y + u.y);
        p[nent] = make_double2(p[nent].x + v.x, p[nent].y + v.y);
    }
}

// Synthesis (ANAL = false): G[order][helicity][row][box] = sum_n U X; analysis: Xd = sum_rows U G.
// Columns of order m >= 0 in four types: (+,m), (-,-m) with U at the row itself, (-,m), (+,-m) with U
// at the mirrored row and (-1)^{n+m}; -m takes (-1)^{m+1}.  Block BT x BT of one type, inner
// step 16, four waves of BT/2 x BT/2.
template <int BT, bool ANAL>
__global__ __launch_bounds__(256) void k_pw_gemm(PwArg a, int ctiles, int accumulate) {
    constexpr int BK = 16, WT = BT / 2, NI = WT / 16, NL = BT * BK / 256;
    const int m = blockIdx.z;
    const int L = a.L;
    const int ty = blockIdx.x / ctiles;
    if (m == 0 && ty >= 2) return;
    const int lo = max(0, a.jlo[m] - a.j0), cnt = a.R2 - lo;
    const int cn = pw_cn(m, L), n0 = m < 1 ? 1 : m;
    const int M = ANAL ? cn : 2 * cnt, K = ANAL ? 2 * cnt : cn;
    const int row0 = blockIdx.y * BT;
    const int NC = 2 * a.nbr;
    const int col0 = (blockIdx.x % ctiles) * BT;
    if (row0 >= M) return;
    if (ANAL && cnt <= 0 && accumulate) return;
    const int ms = (ty & 1) ? -m : m;                 // order of the columns
    const int hel = (ty == 1 || ty == 2) ? 1 : 0;     // 0: +, 1: -
    const bool mir = ty >= 2;
    const double fac = (ty & 1) && !(m & 1) ? -1.0 : 1.0;  // (-1)^{m+1} on -m
    __shared__ double As[BK][BT + 2];
    __shared__ double Bs[BK][BT + 2];
    const double *Um = a.U + pw_ucnt(m, L) * a.ustr;
    auto row_of = [&](int q) { return q < cnt ? lo + q : a.R2 + lo + q - cnt; };
    auto pos_of = [&](int lr) { return lr < a.R2 ? a.a0 + lr : a.a1 + lr - a.R2; };
    auto mirror = [&](int lr) { return lr < a.R2 ? lr + a.R2 : lr - a.R2; };
    const double *Xr = (const double *)(a.X + (2 * pw_xcnt(ms, L) + (int64_t)hel * cn) * a.nbr);
    double *Xw = (double *)(a.Xd + (2 * pw_xcnt(ms, L) + (int64_t)hel * cn) * a.nbr);
    double *Gm = (double *)(a.G + (int64_t)((ms + L) * 2 + hel) * 2 * a.R2 * a.nbr);
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int li = lane & 15, lk = lane >> 4;
    const int wr = (w >> 1) * WT, wc = (w & 1) * WT;
    dv4 acc[NI][NI];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = dv4{0, 0, 0, 0};
    double ra[NL], rb[NL];
    const int cb = min(col0 + (tid & (BT - 1)), NC - 1);
    int64_t arow[ANAL ? NL : 1];
    if constexpr (ANAL) {
#pragma unroll
        for (int e = 0; e < NL; ++e) arow[e] = (int64_t)min(row0 + (tid >> 4) + 16 * e, M - 1) * a.ustr;
    } else {
        arow[0] = pos_of(row_of(min(row0 + (tid & (BT - 1)), M - 1)));
    }
    auto load = [&](int k0) {
#pragma unroll
        for (int e = 0; e < NL; ++e) {
            if constexpr (ANAL) {
                const int k = k0 + (tid & 15);
                const double v = Um[arow[e] + pos_of(row_of(min(k, K - 1)))];
                ra[e] = k < K ? v : 0.0;
            } else {
                const int k = k0 + tid / BT + (256 / BT) * e;
                const double v = Um[(int64_t)min(k, K - 1) * a.ustr + arow[0]];
                ra[e] = k < K ? v : 0.0;
            }
            const int k = min(k0 + tid / BT + (256 / BT) * e, K - 1);
            if constexpr (ANAL) {
                const int lr = row_of(k);
                rb[e] = Gm[(int64_t)(mir ? mirror(lr) : lr) * NC + cb];
            } else {
                const double v = Xr[(int64_t)k * NC + cb];
                rb[e] = mir && ((n0 + k + m) & 1) ? -v : v;
            }
        }
    };
    if (K > 0) load(0);
    for (int k0 = 0; k0 < K; k0 += BK) {
#pragma unroll
        for (int e = 0; e < NL; ++e) {
            const int k = tid / BT + (256 / BT) * e;
            if constexpr (ANAL)
                As[tid & 15][(tid >> 4) + 16 * e] = ra[e];
            else
                As[k][tid & (BT - 1)] = ra[e];
            Bs[k][tid & (BT - 1)] = rb[e];
        }
        __syncthreads();
        if (k0 + BK < K) load(k0 + BK);
#pragma unroll
        for (int kc = 0; kc < BK; kc += 4) {
            double fa[NI], fb[NI];
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                fa[i] = As[kc + lk][wr + 16 * i + li];
                fb[i] = Bs[kc + lk][wc + 16 * i + li];
            }
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int j = 0; j < NI; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[i], fb[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = row0 + wr + 16 * i + 4 * v + lk;
            if (r >= M) continue;
            double f = fac;
            double *o;
            if constexpr (ANAL) {
                if (mir && ((n0 + r + m) & 1)) f = -f;
                o = Xw + (int64_t)r * NC;
            } else {
                const int lr = row_of(r);
                o = Gm + (int64_t)(mir ? mirror(lr) : lr) * NC;
            }
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                const int cidx = col0 + wc + 16 * j + li;
                if (cidx >= NC) continue;
                const double x = f * acc[i][j][v];
                if (ANAL && accumulate)
                    o[cidx] += x;
                else
                    o[cidx] = x;
            }
        }
}

// a / d for 0 <= a < 2^20 from inv = 1 / d in FP32: (a + 1/2) / d is at least 1 / (2 d) from
// the next whole number, 2^-22 a / d the error of the product.
__device__ __forceinline__ int div_small(int a, float inv) { return (int)(((float)a + 0.5f) * inv); }

// Azimuthal transforms of NB boxes of one (row, helicity), in place in LDS: decimation in
// frequency with radices 2, 3, 4, 5 (natural order in, digit-reversed out).  Forward: orders
// -mF..mF of G to azimuths, e^{+i m phi}; inverse: azimuths to orders, e^{-i m phi}.
// Bound by LDS passes, barriers and short pieces of G (waves wait 70% of the time; 64 boxes of order
// 410: 1.09 ms a direction).  Index divisions go through FP32 and the radices are read
// from memory: as integer divisions and a local copy in scratch they took 1.60 ms.
template <bool INV>
__global__ __launch_bounds__(512) void k_pw_fft(PwArg a, int NBmax) {
    extern __shared__ double2 sm[];
    const int lr = blockIdx.y >> 1, hel = blockIdx.y & 1;
    const int node = a.j0 + (lr < a.R2 ? lr : lr - a.R2);
    const PwFft &P = a.fft[a.fftof[node]];
    const int N = P.N, mF = a.mF[node], npass = P.npass;
    const int b0 = blockIdx.x * NBmax;
    const int NB = min(NBmax, a.nbr - b0);
    const int tid = threadIdx.x, nt = blockDim.x;
    const double2 *tw = a.tw + P.tw;
    const int32_t *perm = a.perm + P.perm;
    const int64_t rows = 2 * a.R2;
    double2 *g = a.G + (int64_t)hel * rows * a.nbr + (int64_t)lr * a.nbr + b0;  // + (m + L) 2 rows nbr
    const int64_t gs = 2 * rows * a.nbr;
    const int64_t fb = 2 * a.cpre[lr] * a.nbr + ((int64_t)hel * a.nbr + b0) * N;
    double2 *f = (INV ? a.H : a.F) + fb;
    const float iNB = 1.0f / NB, iN = 1.0f / N;
    if (!INV) {
        // boxes fastest in memory; x[b][i], i = m mod N
        for (int i = tid; i < N * NB; i += nt) {
            const int q = div_small(i, iNB), b = i - q * NB;
            const int m = q <= mF ? q : q - N;  // N > 2 mF
            sm[b * N + q] = m >= -mF ? g[(int64_t)(m + a.L) * gs + b] : make_double2(0.0, 0.0);
        }
    } else {
        for (int i = tid; i < N * NB; i += nt) sm[i] = f[i];
    }
    __syncthreads();
    int M = N;
    for (int ps = 0; ps < npass; ++ps) {
        const int r = P.radix[ps];
        const float ir = 1.0f / r;
        const int S = div_small(M, ir), nbf = div_small(N, ir), step = div_small(N, 1.0f / M);
        const float iS = 1.0f / S, inbf = 1.0f / nbf;
        for (int i = tid; i < nbf * NB; i += nt) {
            const int b = div_small(i, inbf), q = i - b * nbf;
            const int blk = div_small(q, iS), j = q - blk * S;
            double2 *x = sm + b * N + blk * M + j;
            auto twid = [&](int e, double2 v) {
                double2 c = tw[e];
                if (INV) c.y = -c.y;
                return make_double2(c.x * v.x - c.y * v.y, c.x * v.y + c.y * v.x);
            };
            const double sg = INV ? -1.0 : 1.0;
            if (r == 4) {
                const double2 x0 = x[0], x1 = x[S], x2 = x[2 * S], x3 = x[3 * S];
                const double2 s0 = make_double2(x0.x + x2.x, x0.y + x2.y), d0 = make_double2(x0.x - x2.x, x0.y - x2.y);
                const double2 s1 = make_double2(x1.x + x3.x, x1.y + x3.y), d1 = make_double2(x1.x - x3.x, x1.y - x3.y);
                const double2 id = make_double2(-sg * d1.y, sg * d1.x);  // +-i d1
                x[0] = make_double2(s0.x + s1.x, s0.y + s1.y);
                x[S] = twid(step * j, make_double2(d0.x + id.x, d0.y + id.y));
                x[2 * S] = twid(2 * step * j, make_double2(s0.x - s1.x, s0.y - s1.y));
                x[3 * S] = twid(3 * step * j, make_double2(d0.x - id.x, d0.y - id.y));
            } else if (r == 2) {
                const double2 x0 = x[0], x1 = x[S];
                x[0] = make_double2(x0.x + x1.x, x0.y + x1.y);
                x[S] = twid(step * j, make_double2(x0.x - x1.x, x0.y - x1.y));
            } else if (r == 3) {
                const double h = sg * 0.86602540378443864676;
                const double2 x0 = x[0], x1 = x[S], x2 = x[2 * S];
                const double2 s = make_double2(x1.x + x2.x, x1.y + x2.y), d = make_double2(x1.x - x2.x, x1.y - x2.y);
                const double2 c = make_double2(x0.x - 0.5 * s.x, x0.y - 0.5 * s.y), e = make_double2(-h * d.y, h * d.x);
                x[0] = make_double2(x0.x + s.x, x0.y + s.y);
                x[S] = twid(step * j, make_double2(c.x + e.x, c.y + e.y));
                x[2 * S] = twid(2 * step * j, make_double2(c.x - e.x, c.y - e.y));
            } else {
                const double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;
                const double s1 = sg * 0.95105651629515357212, s2 = sg * 0.58778525229247312917;
                const double2 x0 = x[0], x1 = x[S], x2 = x[2 * S], x3 = x[3 * S], x4 = x[4 * S];
                const double2 p = make_double2(x1.x + x4.x, x1.y + x4.y), q1 = make_double2(x1.x - x4.x, x1.y - x4.y);
                const double2 u = make_double2(x2.x + x3.x, x2.y + x3.y), v = make_double2(x2.x - x3.x, x2.y - x3.y);
                const double2 A = make_double2(x0.x + c1 * p.x + c2 * u.x, x0.y + c1 * p.y + c2 * u.y);
                const double2 B = make_double2(x0.x + c2 * p.x + c1 * u.x, x0.y + c2 * p.y + c1 * u.y);
                const double2 E = make_double2(s1 * q1.x + s2 * v.x, s1 * q1.y + s2 * v.y);
                const double2 G = make_double2(s2 * q1.x - s1 * v.x, s2 * q1.y - s1 * v.y);
                x[0] = make_double2(x0.x + p.x + u.x, x0.y + p.y + u.y);
                x[S] = twid(step * j, make_double2(A.x - E.y, A.y + E.x));
                x[2 * S] = twid(2 * step * j, make_double2(B.x - G.y, B.y + G.x));
                x[3 * S] = twid(3 * step * j, make_double2(B.x + G.y, B.y - G.x));
                x[4 * S] = twid(4 * step * j, make_double2(A.x + E.y, A.y - E.x));
            }
        }
        M = S;
        __syncthreads();
    }
    if (!INV) {
        for (int i = tid; i < N * NB; i += nt) {
            const int b = div_small(i, iN), q = i - b * N;
            f[i] = sm[b * N + perm[q]];
        }
    } else {
        const int nm = 2 * mF + 1;
        for (int i = tid; i < nm * NB; i += nt) {
            const int qm = div_small(i, iNB), b = i - qm * NB, m = qm - mF;
            g[(int64_t)(m + a.L) * gs + b] = sm[b * N + perm[m < 0 ? m + N : m]];
        }
    }
}

// H(target) = sum over its sources of T F: wave per (row, 64 azimuths, parent), the eight
// children's sums of both helicities in registers; a source's samples are read once per
// parent, the tables by neighbouring waves of the same azimuths from one L2 (mixed precision
// reads them rounded to FP32, half of the bytes; samples and sums stay FP64).
// Bound by the reads of tables and samples, through L1 from L2 (16 bytes of table per 16 flops): 16.4
// TB/s of L2 reads at orders 97 and 174, 16.1 at order 410, where HBM delivers 6.3 of them (25 GB
// a launch for 2.1 GB of samples and 0.6 GB of tables: the dies fetch both several times).  The loads of a
// source and all eight children are in flight while the previous source's products run, also
// for children that the source does not reach (they read some entry of the first table): with
// a branch around each load every product waited for its own load.  56046 translations of
// orders 97 and 174: 9.5 ms with loads behind branches, 7.2 with a source's loads first and
// the next source's beside the products, 5.2 as here with 32-bit offsets from scalar row
// addresses.
template <typename TT>
__global__ __launch_bounds__(256) void k_pw_m2l(const TT *__restrict__ T, PwArg a, const PwParent *__restrict__ par, int npar,
                                                const PwSource *__restrict__ src, const PwMaps *__restrict__ map,
                                                int nb, int ptiles, int64_t nblocks) {
    const int64_t id = die_order(blockIdx.x, nblocks);
    const int pt = (int)(id % ptiles);
    const int at = (int)(id / ptiles);
    const int lr = blockIdx.y;
    const int node = a.j0 + (lr < a.R2 ? lr : lr - a.R2);
    const int N = a.N[node];
    if (at * 64 >= N) return;
    const int p = __builtin_amdgcn_readfirstlane(pt * 4 + (int)(threadIdx.x >> 6));
    if (p >= npar) return;
    const int lane = threadIdx.x & 63;
    const int i0 = at * 64 + lane;
    const int i = min(i0, N - 1);
    const int rhs = blockIdx.z;
    const int mlr = lr < a.R2 ? lr + a.R2 : lr - a.R2;
    const int64_t t0 = a.tpre[lr < a.R2 ? a.a0 + lr : a.a1 + lr - a.R2];
    const int64_t t1 = a.tpre[mlr < a.R2 ? a.a0 + mlr : a.a1 + mlr - a.R2];
    const int64_t fb = 2 * a.cpre[lr] * a.nbr;
    const double2 *Fp = a.F + fb + (int64_t)rhs * nb * N + i;
    const double2 *Fm = Fp + (int64_t)a.nbr * N;
    const PwParent P = par[p];
    double2 hp[8], hm[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) hp[c] = hm[c] = make_double2(0.0, 0.0);
    // azimuth i of a child's table: +-(i - quarter N / 4) mod N, in bytes from the row's start
    const int nB = N * (int)sizeof(TT), n4B = (N >> 2) * (int)sizeof(TT);
    const uint32_t tB = (uint32_t)(a.tsn * sizeof(TT));
    const char *r0 = (const char *)(T + t0), *r1 = (const char *)(T + t1);
    auto load_T = [&](const PwMaps &M, TT tv[8]) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const PwMap q = M.child[c];
            const uint32_t o = (uint32_t)(__mul24(i, q.sign * (int)sizeof(TT)) + q.shift * n4B);
            const char *row = (q.flip ? r1 : r0) + (uint64_t)(uint32_t)q.table * tB;
            tv[c] = *(const TT *)(row + min(o, o + (uint32_t)nB));
        }
    };
    auto product = [&](const PwSource &S, const TT tv[8], double2 fp, double2 fm) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            if (!(S.mask >> c & 1)) continue;
            const double2 t = make_double2(tv[c].x, tv[c].y);
            hp[c].x = fma(t.x, fp.x, hp[c].x);
            hp[c].x = fma(-t.y, fp.y, hp[c].x);
            hp[c].y = fma(t.x, fp.y, hp[c].y);
            hp[c].y = fma(t.y, fp.x, hp[c].y);
            hm[c].x = fma(t.x, fm.x, hm[c].x);
            hm[c].x = fma(-t.y, fm.y, hm[c].x);
            hm[c].y = fma(t.x, fm.y, hm[c].y);
            hm[c].y = fma(t.y, fm.x, hm[c].y);
        }
    };
    if (P.beg < P.end) {
        // two sources in flight: the tables' and samples' loads of one during the products of
        // the other; a source's map is read one source ahead of its loads
        PwSource S[2], S1 = src[P.beg], S2 = src[min(P.beg + 1, P.end - 1)];
        PwMaps M1 = map[S1.r];
        double2 fp[2], fm[2];
        TT tv[2][8];
        auto load = [&](int e, int q) {
            S[q] = S1;
            fp[q] = Fp[(int64_t)S1.box * N];
            fm[q] = Fm[(int64_t)S1.box * N];
            load_T(M1, tv[q]);
            M1 = map[S2.r];
            S1 = S2;
            S2 = src[min(e + 2, P.end - 1)];
        };
        load(P.beg, 0);
        int e = P.beg;
        for (; e + 1 < P.end; e += 2) {
            load(e + 1, 1);
            product(S[0], tv[0], fp[0], fm[0]);
            load(min(e + 2, P.end - 1), 0);
            product(S[1], tv[1], fp[1], fm[1]);
        }
        if (e < P.end) product(S[0], tv[0], fp[0], fm[0]);
    }
    if (i0 >= N) return;
    double2 *Hp = a.H + fb + (int64_t)rhs * nb * N + i;
    double2 *Hm = Hp + (int64_t)a.nbr * N;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        if (P.child[c] < 0) continue;
        Hp[(int64_t)P.child[c] * N] = hp[c];
        Hm[(int64_t)P.child[c] * N] = hm[c];
    }
}

void launch_pw_utable(int L, int Q2, int j0, int R2, int a0, int a1, int64_t ustr, const double *mu, double *U,
                      hipStream_t s) {
    hipLaunchKernelGGL(k_pw_utable, dim3((2 * R2 + 63) / 64, L + 1), dim3(64), 0, s, L, Q2, j0, R2, a0, a1, ustr, mu, U);
}
void launch_pw_hankel(int ncanon, int P, const double *t, const int32_t *terms, double2 *h, hipStream_t s) {
    hipLaunchKernelGGL(k_pw_hankel, dim3(ncanon), dim3(64), 0, s, P, t, terms, h);
}
void launch_pw_ttable(int ncanon, int P, int Q2, int j0, int R2, int a0, int a1, int maxN, const double *mu,
                      const double *canon, const int32_t *N, const int64_t *tpre, int64_t tsn, const double2 *h,
                      double2 *T, float2 *T32, hipStream_t s) {
    hipLaunchKernelGGL(k_pw_ttable, dim3((maxN + 255) / 256, 2 * R2, ncanon), dim3(256), sizeof(double2) * (P + 1), s,
                       P, Q2, j0, R2, a0, a1, mu, canon, N, tpre, tsn, h, T, T32);
}
void launch_pw_pack(const PwArg &a, int nb, int64_t off, const double2 *C, int64_t stride, hipStream_t s) {
    hipLaunchKernelGGL(k_pw_pack, dim3((a.L * (a.L + 2) + 15) / 16, (a.nbr + 31) / 32), dim3(256), 0, s, a, nb, off, C,
                       stride);
}
void launch_pw_unpack(const PwArg &a, int nb, int64_t off, double2 *D, int64_t stride, hipStream_t s) {
    hipLaunchKernelGGL(k_pw_unpack, dim3((a.L * (a.L + 2) + 15) / 16, (a.nbr + 31) / 32), dim3(256), 0, s, a, nb, off,
                       D, stride);
}
void launch_pw_synth(const PwArg &a, hipStream_t s) {
    const int ct = (2 * a.nbr + 63) / 64;
    hipLaunchKernelGGL((k_pw_gemm<64, false>), dim3(4 * ct, (2 * a.R2 + 63) / 64, a.L + 1), dim3(256), 0, s, a, ct, 0);
}
void launch_pw_anal(const PwArg &a, int accumulate, hipStream_t s) {
    const int ct = (2 * a.nbr + 63) / 64;
    hipLaunchKernelGGL((k_pw_gemm<64, true>), dim3(4 * ct, (a.L + 63) / 64, a.L + 1), dim3(256), 0, s, a, ct,
                       accumulate);
}
void launch_pw_fft(const PwArg &a, int inverse, int maxN, hipStream_t s) {
    // boxes per block: what 64 KiB of LDS holds, at most 8 (128-byte pieces of G).  64 boxes of
    // order 410: 1.09 ms; in 40 or 27 KiB 1.18 and 1.29; with 256 or 1024 threads 1.40 and 1.42
    const int NB = std::max(1, std::min(8, 65536 / (16 * maxN)));
    const dim3 grid((a.nbr + NB - 1) / NB, 4 * a.R2);
    const size_t shm = 16 * (size_t)NB * maxN;
    if (inverse)
        hipLaunchKernelGGL(k_pw_fft<true>, grid, dim3(512), shm, s, a, NB);
    else
        hipLaunchKernelGGL(k_pw_fft<false>, grid, dim3(512), shm, s, a, NB);
}
void launch_pw_m2l(const PwArg &a, const PwParent *par, int npar, const PwSource *src, const PwMaps *map, int nb,
                   int nrhs, int maxN, hipStream_t s) {
    const int ptiles = (npar + 3) / 4;
    const int64_t nblocks = (int64_t)ptiles * ((maxN + 63) / 64);
    const dim3 grid((unsigned)nblocks, 2 * a.R2, nrhs);
    if (a.T32)
        hipLaunchKernelGGL(k_pw_m2l<float2>, grid, dim3(256), 0, s, a.T32, a, par, npar, src, map, nb, ptiles, nblocks);
    else
        hipLaunchKernelGGL(k_pw_m2l<double2>, grid, dim3(256), 0, s, a.T, a, par, npar, src, map, nb, ptiles, nblocks);
}

}  // namespace ifs
