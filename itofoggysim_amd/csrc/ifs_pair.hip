// Sphere-pair translations with matrices shared by every pair (gfx950).
//
// A translation rotates the source so that z points along the pair, shifts it along z
// and rotates back.  With per-pair Wigner and coaxial tables (about 30 L^3 bytes) that is
// bound by reading the tables; here every matrix is common to all pairs and only O(L)
// numbers belong to one pair:
//
//   rotation   d^n(theta)_{km} = i^k sum_j D_jk e^{-ij theta} D_jm (-i)^m,  D = d^n(pi/2):
//              two products with the fixed D and diagonal phases.  D_{j,-m} = (-1)^{n+j}
//              D_jm and D_{-j,m} = (-1)^{n+m} D_jm split each product into four blocks by
//              the parities of j and m, half the work of a full one, so the two together
//              cost what one rotation with a table of d^n(theta) does.
//   shift      P_m(n,nu) = sqrt((2n+1)(2nu+1))/2 int d^n_{m,1} d^nu_{m,1} T dmu (Q_m: d_{m,-1}),
//              T(mu) = sum_{p <= Ls+Lt} i^p (2p+1) h1_p(t) P_p(mu): a product to the
//              Gauss-Legendre nodes, the pair's T at the nodes, a product back.
//
// Four pairs of one target make the 16 real columns of a matrix-core tile.  The FP64
// tile D(16x16) += A(16x4) B(4x16) holds D[4v + l/16][l%16] in value v of lane l and
// takes B[l/16][l%16] from lane l, so value v of one product's result is the B operand
// of inner step v of the next: the chained products stay in registers, without LDS.
//
// The quadrature sum carries rounding of the largest |h1_p|, so pairs closer than
// t/2-growth allows (PairTile::Q = 0, rule in ifs_pair.cpp) take coaxial tables from
// the degree recurrence instead; their rotations run here all the same.
//
// Bound by the latency of operand loads: the matrix cores are busy 28 to 35% of the time, with
// 3.4 to 6.2 waves resident on a SIMD that wait 33 to 63% of theirs (tiles are 50-75% full at orders
// 10 to 25).  Against per-pair tables: 22650 pairs of orders 10-18 (151 spheres at
// 800 nm) 3.57 -> 0.47 ms per product, the near field of 2500 spheres at 550 nm (248818
// pairs, orders 9-23) 40.1 -> 7.3 ms, with four right-hand sides (114758 pairs) 81.9 ->
// 13.0 ms; error against 64-bit sums unchanged (3e-13, 1.1e-13).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <math.h>

#include "ifs_pair.h"

namespace ifs {

namespace {

typedef double dv4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ dv4 mma(double a, double b, dv4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
// doubles before degree n in the operand-ordered D: sum_{i<n} 256 rt(i) ks(i)
__device__ __forceinline__ int delta_off(int n) {
    // ks(i) = (i/2 + 4) / 4: 1 for i = 1..., steps of 8 degrees; sum_{i=1}^{n-1} ks(i)
    auto ksum = [](int e) {  // sum_{i=0}^{e-1} ((i >> 1) + 4) >> 2
        const int b = e >> 3, r = e & 7;  // ((i >> 1) + 4) >> 2 = (i >> 3) + 1
        return 8 * (b * (b + 1) / 2) + r * (b + 1);
    };
    int s = ksum(n) - ksum(1);
    if (n > 32) s += ksum(n) - ksum(32);  // two row tiles from degree 32 on
    return 256 * s;
}
__device__ __forceinline__ int yrow(int n, int k, int K) { return (int)rows_off(n, K) + k + (n < K ? n : K); }

}  // namespace

// One degree of the three-term recurrence of d^n_{k,m} at x = cos(beta).
__device__ __forceinline__ double wig_next(int n, double k, double m, double x, double d1, double d2) {
    const double nn = n, n1 = nn - 1.0;
    return ((2.0 * nn - 1.0) * (nn * n1 * x - k * m) * d1 -
            nn * sqrt((n1 * n1 - k * k) * (n1 * n1 - m * m)) * d2) /
           (n1 * sqrt((nn * nn - k * k) * (nn * nn - m * m)));
}

// d^n_{jm}(pi/2), n = j..NL, of block j and thread m <= j, and its transpose, into the
// operand order of the rotations.  Seed d^j_{jm} = (-1)^{j-m} 2^{-j} sqrt(binomial(2j, j+m)).
__global__ void k_pair_delta(int NL, double *__restrict__ delta) {
    const int j = blockIdx.x, m = threadIdx.x;
    if (m > j) return;
    double c = 1.0;
    for (int i = j; i > m; --i) c = c * (double)(j + i) / (double)(j - i + 1);
    const double sg = ((j - m) & 1) ? -1.0 : 1.0;
    double d2 = 0.0, d1 = sg * ldexp(sqrt(c), -j);
    auto put = [&](int n, int r_, int c_, double v) {
        const int r = r_ >> 1, q = c_ >> 1, rt = pair_rt(n), ks = pair_ks(n);
        delta[delta_off(n) + ((((r_ & 1) * 2 + (c_ & 1)) * rt + (r >> 4)) * ks + (q >> 2)) * 64 + (r & 15) +
              16 * (q & 3)] = v;
    };
    for (int n = j; n <= NL; ++n) {
        if (n > j) {
            // n = 1 (j = m = 0): d^1_00(pi/2) = 0
            const double d = n == 1 ? 0.0 : wig_next(n, j, m, 0.0, d1, d2);
            d2 = d1;
            d1 = d;
        }
        if (n < 1) continue;
        put(n, j, m, d1);
        if (m < j) put(n, m, j, sg * d1);
    }
}

// Matrices of one node set: block (m, +-1), thread per node.  U_n = sqrt((2n+1)/2) d^n_{m,+-1}.
__global__ void k_pair_quad(int NL, int Q, const double *__restrict__ mu, double *__restrict__ mats) {
    const int m = blockIdx.x, ty = blockIdx.y, q = threadIdx.x;
    const double x = mu[q], s = ty == 0 ? 1.0 : -1.0;
    const double ch = sqrt(0.5 * (1.0 + x)), sh = sqrt(0.5 * (1.0 - x));
    const int QT = Q >> 4, S1 = (NL + 3) / 4, UT = (NL + 15) / 16;
    double *A1 = mats + (int64_t)(m * 2 + ty) * QT * S1 * 64;
    double *A2 = mats + (int64_t)(NL + 1) * 2 * QT * S1 * 64 + (int64_t)(m * 2 + ty) * UT * 4 * QT * 64;
    const int q0 = m < 1 ? 1 : m;
    // seeds: d^m_{m,s} = sqrt((2m)!/((m+1)!(m-1)!)) ch^{m+s} (-sh)^{m-s}, d^1_{0,s} = s sin/sqrt(2)
    double d1;
    if (m == 0) {
        d1 = s * sqrt(2.0) * ch * sh;
    } else {
        double c = 1.0;  // (2m)! / ((m+1)! (m-1)!) 4^{-(m-1)}, (2 ch sh)^{m-1}
        double p = 1.0;
        for (int i = 2; i <= m; ++i) {
            c *= (double)(2 * i) * (double)(2 * i - 1) / (4.0 * (double)(i + 1) * (double)(i - 1));
            p *= -2.0 * ch * sh;
        }
        d1 = sqrt(c) * p * (ty == 0 ? ch * ch : sh * sh);
    }
    double d2 = 0.0;
    for (int n = q0; n <= NL; ++n) {
        if (n > q0) {
            const double d = wig_next(n, m, s, x, d1, d2);
            d2 = d1;
            d1 = d;
        }
        const double u = sqrt(n + 0.5) * d1;
        const int i = n - q0;
        A1[((int64_t)(q >> 4) * S1 + (i >> 2)) * 64 + (q & 15) + 16 * (i & 3)] = u;
        A2[((int64_t)(i >> 4) * 4 * QT + (q >> 2)) * 64 + (i & 15) + 16 * (q & 3)] = u;
    }
}

// Per pair: the phase rows and the weighted T at the nodes.  Block per slot.
__global__ void k_pair_tables(const PairTile *__restrict__ tiles, const PairSlot *__restrict__ slots, int t0,
                              const double *__restrict__ quad, double2 *__restrict__ tab) {
    extern __shared__ double2 h[];
    const int it = t0 + (blockIdx.x >> 2), sl = blockIdx.x & 3;
    const PairTile T = tiles[it];
    const PairSlot S = slots[4 * it + sl];
    double2 *o = tab + T.off_tab + (int64_t)sl * T.tabw;
    const double theta = acos(S.cth);
    for (int m = threadIdx.x; m <= T.NL; m += blockDim.x) {
        double sn, cs;
        sincos((double)m * S.phi, &sn, &cs);  // times (-i)^m
        switch (m & 3) {
            case 0: o[m] = make_double2(cs, sn); break;
            case 1: o[m] = make_double2(sn, -cs); break;
            case 2: o[m] = make_double2(-cs, -sn); break;
            default: o[m] = make_double2(-sn, cs);
        }
        sincos((double)m * theta, &sn, &cs);
        o[T.NL + 1 + m] = make_double2(cs, -sn);
    }
    if (T.Q == 0) return;
    const int P = S.Ls + T.Lt;
    if (threadIdx.x == 0) {
        // h1_p(t), p = 0..P: j by Miller's downward recurrence, y upward
        const double x = S.t;
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
        for (int n = 0; n <= P; ++n) {
            h[n].x *= scale;
            h[n].y = ym1;
            const double yn = (2.0 * n + 3.0) / x * y - ym1;
            ym1 = y;
            y = yn;
        }
    }
    __syncthreads();
    const double *mu = quad + T.off_mu, *w = mu + T.Q;
    for (int q = threadIdx.x; q < T.Q; q += blockDim.x) {
        const double x = mu[q];
        double pm1 = 0.0, pc = 1.0, ar = 0.0, ai = 0.0;
        for (int p = 0; p <= P; ++p) {
            const double f = (2.0 * p + 1.0) * pc;
            const double2 c = h[p];
            switch (p & 3) {  // i^p h_p
                case 0: ar += f * c.x, ai += f * c.y; break;
                case 1: ar -= f * c.y, ai += f * c.x; break;
                case 2: ar -= f * c.x, ai -= f * c.y; break;
                default: ar += f * c.y, ai -= f * c.x;
            }
            const double pn = ((2.0 * p + 1.0) * x * pc - p * pm1) / (p + 1.0);
            pm1 = pc;
            pc = pn;
        }
        o[2 * (T.NL + 1) + q] = make_double2(w[q] * ar, w[q] * ai);
    }
}

// The D operands of one degree, [a][b][row tile][inner step]: loaded once per wave, used by
// both products (and by every tile of a segment).  KS: inner steps, (n >> 3) + 1.
template <int RT, int KS>
struct DFrag {
    double d[2][2][RT][KS];
    __device__ __forceinline__ void load(const double *__restrict__ D, int lane) {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int r = 0; r < RT; ++r)
#pragma unroll
                    for (int s = 0; s < KS; ++s) d[a][b][r][s] = D[(((a * 2 + b) * RT + r) * KS + s) * 64 + lane];
    }
};

// The two D products of a rotation of degree n on one tile of columns: load(b, c, p, q)
// gives u_m + u_-m and u_m - u_-m of inner class b at m = b + 2c (this lane's column);
// on return vp[a][i], vm[a][i] (i = 4 rt + v) are the results at +-(a + 2r), r = 16 rt +
// 4 v + l/16, without the outer phases.  th: e^{-ij theta} of this lane's pair.  The
// inner steps are unrolled: all loads of a step chain are in flight before its products.
template <int RT, int KS, typename Load>
__device__ __forceinline__ void rotate(int n, const DFrag<RT, KS> &D, const double2 *__restrict__ th, int lane,
                                       Load load, double (&vp)[2][4 * RT], double (&vm)[2][4 * RT]) {
    const int lk = lane >> 4;
    const double sg = (lane & 1) ? -1.0 : 1.0;   // im lane
    const double sn = (n & 1) ? -1.0 : 1.0;
    const bool odd = n & 1;
    double e[KS][2], o[KS][2];
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            double p, q;
            load(b, 4 * s + lk, p, q);
            e[s][b] = odd ? q : p;  // n + a even takes p
            o[s][b] = odd ? p : q;
        }
    dv4 acc[2][2][RT];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < RT; ++r) acc[a][b][r] = dv4{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                acc[0][b][r] = mma(D.d[0][b][r][s], e[s][b], acc[0][b][r]);
                acc[1][b][r] = mma(D.d[1][b][r][s], o[s][b], acc[1][b][r]);
            }
    // inner step s of the second product is value v = s % 4 of row tile s / 4: the first KS
    // values hold all of n
    double P[2][KS], Q[2][KS];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int j = a + 2 * (4 * s + lk);
            const double A = acc[a][0][s >> 2][s & 3], B = acc[a][1][s >> 2][s & 3];
            const double x = A + B, y = sn * (A - B);       // v_j, v_-j
            const double2 f = th[j < n ? j : n];            // cos, -sin
            const double xo = __shfl_xor(x, 1, 64), yo = __shfl_xor(y, 1, 64);
            // e^{-ij theta} v_j and e^{ij theta} v_-j: this lane's part from both
            const double wp = f.x * x - sg * f.y * xo;
            const double wm = f.x * y + sg * f.y * yo;
            P[a][s] = j == 0 ? wp : wp + wm;
            Q[a][s] = j == 0 ? 0.0 : wp - wm;
        }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < RT; ++r) acc[a][b][r] = dv4{0, 0, 0, 0};
    // D_jk = (-1)^{j+k} D_kj: the same operands, minus where the parities differ
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const double ev = odd ? Q[b][s] : P[b][s], ov = odd ? P[b][s] : Q[b][s];
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                acc[0][b][r] = mma(D.d[0][b][r][s], ev, acc[0][b][r]);
                acc[1][b][r] = mma(D.d[1][b][r][s], ov, acc[1][b][r]);
            }
        }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const double A = a == 0 ? acc[a][0][r][v] : -acc[a][0][r][v];
                const double B = a == 0 ? -acc[a][1][r][v] : acc[a][1][r][v];
                vp[a][4 * r + v] = A + B;
                vm[a][4 * r + v] = sn * (A - B);
            }
}

// Forward rotation: wave per (tile, degree), x -> Y.
template <int RT, int KS>
__device__ __forceinline__ void pair_fwd(int n, const PairTile &T, const PairSlot *__restrict__ slots,
                                         const double *__restrict__ delta, const double2 *__restrict__ tab,
                                         const double2 *__restrict__ src, double *__restrict__ y) {
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const int part = li & 3;
    DFrag<RT, KS> D;
    D.load(delta + delta_off(n), lane);
    const PairSlot S = slots[li >> 2];
    const double2 *ph = tab + T.off_tab + (int64_t)(li >> 2) * T.tabw;
    const double2 *th = ph + T.NL + 1;
    const bool live = S.src >= 0 && n <= S.Ls;
    const double2 *xa = src + (live ? S.src + n * n - 1 + n : 0);
    const double2 *xb = xa + (live ? (int64_t)S.Ls * (S.Ls + 2) : 0);
    const double s2 = part < 2 ? 1.0 : -1.0;
    const bool im = part & 1;
    double vp[2][4 * RT], vm[2][4 * RT];
    rotate<RT, KS>(n, D, th, lane,
                   [&](int b, int c, double &p, double &q) {
                       const int m = b + 2 * c;
                       if (!live || m > n) {
                           p = q = 0.0;
                           return;
                       }
                       const double2 f = ph[m], a0 = xa[m], b0 = xb[m], a1 = xa[-m], b1 = xb[-m];
                       const double xr = a0.x + s2 * b0.x, xi = a0.y + s2 * b0.y;
                       const double yr = a1.x + s2 * b1.x, yi = a1.y + s2 * b1.y;
                       const double up = im ? f.x * xi + f.y * xr : f.x * xr - f.y * xi;
                       const double um = im ? f.x * yi - f.y * yr : f.x * yr + f.y * yi;
                       p = m == 0 ? up : up + um;
                       q = m == 0 ? 0.0 : up - um;
                   },
                   vp, vm);
    const int K = T.K;
    const int row = yrow(n, 0, K);
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int i = 0; i < KS; ++i) {
            const int r = 4 * i + lk;
            const int k = a + 2 * r;
            if (k > n || k > K) continue;
            const double sr = (r & 1) ? -1.0 : 1.0;
            if (a == 0) {  // i^{+-k} = (-1)^r
                y[(int64_t)(row + k) * 16 + li] = sr * vp[a][i];
                if (k > 0) y[(int64_t)(row - k) * 16 + li] = sr * vm[a][i];
            } else {  // i^k = i (-1)^r, i^{-k} = -i (-1)^r: the parts change places
                const double f = im ? -sr : sr;
                y[(int64_t)(row + k) * 16 + (li ^ 1)] = f * vp[a][i];
                y[(int64_t)(row - k) * 16 + (li ^ 1)] = -f * vm[a][i];
            }
        }
}

// RT = 1: degrees 1..31, RT = 2: 32..63.  KSM: the most inner steps that the launch meets.  The
// operands of KSM steps set the registers (forward / backward 67 / 127 for two, 84 / 165 for
// three, 114 / 219 for four) and so the waves that hide the loads, which bound both kernels:
// each range of degrees has a launch of its own.
template <int RT, int KSM>
__global__ __launch_bounds__(256) void k_pair_fwd(const PairTile *__restrict__ tiles,
                                                  const PairSlot *__restrict__ slots, int t0, int ntiles, int n0,
                                                  const double *__restrict__ delta, const double2 *__restrict__ tab,
                                                  const double2 *__restrict__ src, int64_t src_stride,
                                                  double *__restrict__ Y, int64_t y_stride) {
    const int ti = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    if (ti >= ntiles) return;
    const PairTile T = tiles[t0 + ti];
    const int n = n0 + blockIdx.y;
    if (n > T.Ls) return;
    const PairSlot *sl = slots + 4 * (t0 + ti);
    const double2 *x = src + blockIdx.z * src_stride;
    double *y = Y + blockIdx.z * y_stride + T.off_y;
    switch (n >> 3) {
        case 4 * (RT - 1): pair_fwd<RT, 4 * RT - 3>(n, T, sl, delta, tab, x, y); break;
        case 4 * (RT - 1) + 1: pair_fwd<RT, 4 * RT - 2>(n, T, sl, delta, tab, x, y); break;
        case 4 * (RT - 1) + 2:
            if constexpr (KSM > 4 * RT - 2) pair_fwd<RT, 4 * RT - 1>(n, T, sl, delta, tab, x, y);
            break;
        default:
            if constexpr (KSM > 4 * RT - 1) pair_fwd<RT, 4 * RT>(n, T, sl, delta, tab, x, y);
    }
}

// Coaxial shift: wave per (tile, order m), Y -> Z at k = +-m.  z_+(m) and z_-(-m) take
// P_m, z_+(-m) and z_-(m) take Q_m, so each of the two products has 16 columns.  The tiles
// of a block share one node set: its matrices pass through LDS one node tile at a time (read
// per wave from L1 they took 8 cache accesses per 64-cycle product and bounded the kernel:
// 5740 tiles of orders 10-18 in 343 us; through LDS, rows read whole, 238 us).  A wave fetches
// its rows of the next node tile while the block works on this one, and a block's tiles have
// similar orders (few waves without work at high m): 48 clusters 588 -> 522 us, 5740 tiles 234.
// Node-set matrices at off_q: for [m][P, Q]: A1[Q/16][S1][64] (rows
// nodes, inner degrees) and after all of them A2[UT][Q/4][64] (rows degrees, inner nodes).
// KS, UT: inner steps of four source degrees and tiles of 16 target degrees that the launch holds.
template <int UT, int KS, int NW>
__global__ __launch_bounds__(64 * NW) void k_pair_axial(const PairTile *__restrict__ tiles,
                                                    const PairSlot *__restrict__ slots,
                                                    const PairGroup *__restrict__ groups,
                                                    const int32_t *__restrict__ order, int NL,
                                                    const double *__restrict__ quad, const double2 *__restrict__ tab,
                                                    const double2 *__restrict__ wax, const double *__restrict__ Y,
                                                    int64_t y_stride, double *__restrict__ Z, int64_t z_stride) {
    constexpr int AR = 2 * KS + 8 * UT, PF = (AR + NW - 1) / NW;
    __shared__ double As[2][AR][64];  // [buffer][type][step] of A1, then [type][t][v] of A2
    const PairGroup G = groups[blockIdx.x];
    const int m = blockIdx.y;
    if (m > G.K) return;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const int ti = order[G.first + (wv < G.count ? wv : 0)];
    const PairTile T = tiles[ti];
    const bool live = wv < G.count && m <= T.K;
    const int K = T.K, Ls = T.Ls, Lt = T.Lt;
    const int q0 = m < 1 ? 1 : m;
    const double *y = Y + blockIdx.z * y_stride + T.off_y;
    double *z = Z + blockIdx.z * z_stride + T.off_z;
    if (G.Q == 0) {
        if (!live) return;
        // close pairs: 16 target degrees of each of the four slots at a time, from their own
        // tables, which hold P(nu, n) = P(n, nu) with the target degree running fastest
        const PairSlot S = slots[4 * ti + lk];
        const int ncol = Lt - q0 + 1;
        const bool on = S.src >= 0 && m <= S.K;
        const double2 *Pb = wax + S.off_ax + (on ? ax_off(m, S.Ls, Lt, S.K) : 0) - q0;
        const double2 *Qb = Pb + (on ? ax_block(m, S.Ls, Lt) : 0);
        for (int n = q0 + li; n <= Lt; n += 16) {
            double zr[4] = {0, 0, 0, 0}, zi[4] = {0, 0, 0, 0};  // z_+(m), z_-(m), z_+(-m), z_-(-m)
            if (on) {
                for (int nu = q0; nu <= S.Ls; ++nu) {
                    const double2 pv = Pb[(nu - q0) * ncol + n], qv = Qb[(nu - q0) * ncol + n];
                    const double2 *yp = (const double2 *)(y + (int64_t)yrow(nu, m, K) * 16 + 4 * lk);
                    const double2 *ym = (const double2 *)(y + (int64_t)yrow(nu, -m, K) * 16 + 4 * lk);
                    const double2 v[4] = {yp[0], yp[1], ym[0], ym[1]};
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const double2 c = (i == 0 || i == 3) ? pv : qv;
                        zr[i] += c.x * v[i].x - c.y * v[i].y;
                        zi[i] += c.x * v[i].y + c.y * v[i].x;
                    }
                }
            }
            double2 *zp = (double2 *)(z + (int64_t)yrow(n, m, K) * 16 + 4 * lk);
            double2 *zm = (double2 *)(z + (int64_t)yrow(n, -m, K) * 16 + 4 * lk);
            zp[0] = make_double2(zr[0], zi[0]);
            zp[1] = make_double2(zr[1], zi[1]);
            if (m > 0) {
                zm[0] = make_double2(zr[2], zi[2]);
                zm[1] = make_double2(zr[3], zi[3]);
            }
        }
        return;
    }
    const bool plus = (li & 3) < 2;  // a part of x_+
    const double sg = (li & 1) ? 1.0 : -1.0;
    const double2 *tq = tab + T.off_tab + (int64_t)(li >> 2) * T.tabw + 2 * (T.NL + 1);
    const int QT = G.Q >> 4, S1 = (NL + 3) / 4, UTN = (NL + 15) / 16;
    const double *A1 = quad + G.off_q + (int64_t)m * 2 * QT * S1 * 64;
    const double *A2 = quad + G.off_q + (int64_t)(NL + 1) * 2 * QT * S1 * 64 + (int64_t)m * 2 * UTN * 4 * QT * 64;
    const int ks = live ? (Ls - q0 + 4) / 4 : 0, ut = live ? (Lt - q0 + 16) / 16 : 0;
    const int ksg = min((G.Ls - q0 + 4) / 4, KS), utg = min((G.Lt - q0 + 16) / 16, UT);  // of the block
    // the source columns stay in registers for all node tiles
    double bp[KS], bq[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        bp[s] = bq[s] = 0.0;
        if (s < ks) {
            const int nu = q0 + 4 * s + lk;
            const int row = yrow(nu <= Ls ? nu : Ls, 0, K);
            double a = y[(int64_t)(row + m) * 16 + li], b = y[(int64_t)(row - m) * 16 + li];
            a = nu <= Ls ? a : 0.0;
            b = nu <= Ls ? b : 0.0;
            bp[s] = plus ? a : b;
            bq[s] = plus ? b : a;
        }
    }
    dv4 u[2][UT];
#pragma unroll
    for (int t = 0; t < UT; ++t) u[0][t] = u[1][t] = dv4{0, 0, 0, 0};
    // a wave stages rows wv, wv + NW, ...: in registers while the block works on the other buffer
    double2 tv[4];
    double pre[PF];
    auto fetch = [&](int qt) {
#pragma unroll
        for (int i = 0; i < PF; ++i) {
            const int r = wv + NW * i;
            pre[i] = 0.0;
            if (r < 2 * KS) {
                const int ty = r >= KS, s = r - ty * KS;
                if (s < ksg) pre[i] = A1[(int64_t)((ty * QT + qt) * S1 + s) * 64 + lane];
            } else if (r < AR) {
                const int q = r - 2 * KS, ty = q >= 4 * UT, t = (q >> 2) - ty * UT;
                if (t < utg) pre[i] = A2[((int64_t)(ty * UTN + t) * 4 * QT + 4 * qt + (q & 3)) * 64 + lane];
            }
        }
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int i = 0; i < PF; ++i)
            if (wv + NW * i < AR) As[buf][wv + NW * i][lane] = pre[i];
    };
    fetch(0);
    stage(0);
    __syncthreads();
    for (int qt = 0; qt < QT; ++qt) {
        const double(*A)[64] = As[qt & 1];
        if (live)
#pragma unroll
            for (int v = 0; v < 4; ++v) tv[v] = tq[16 * qt + 4 * v + lk];
        if (qt + 1 < QT) fetch(qt + 1);
        if (live) {
            dv4 g[2] = {dv4{0, 0, 0, 0}, dv4{0, 0, 0, 0}};
#pragma unroll
            for (int s = 0; s < KS; ++s)
                if (s < ks) {
                    g[0] = mma(A[s][lane], bp[s], g[0]);
                    g[1] = mma(A[KS + s][lane], bq[s], g[1]);
                }
#pragma unroll
            for (int v = 0; v < 4; ++v)
#pragma unroll
                for (int ty = 0; ty < 2; ++ty) {
                    const double x = g[ty][v], xo = __shfl_xor(x, 1, 64);
                    const double b = tv[v].x * x + sg * tv[v].y * xo;
#pragma unroll
                    for (int t = 0; t < UT; ++t)
                        if (t < ut) u[ty][t] = mma(A[2 * KS + (ty * UT + t) * 4 + v][lane], b, u[ty][t]);
                }
        }
        if (qt + 1 < QT) stage((qt + 1) & 1);
        __syncthreads();
    }
    if (!live) return;
#pragma unroll
    for (int t = 0; t < UT; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int n = q0 + 16 * t + 4 * v + lk;
            if (n > Lt) continue;
            const int row = yrow(n, 0, K);
            z[(int64_t)(row + m) * 16 + li] = plus ? u[0][t][v] : u[1][t][v];
            if (m > 0) z[(int64_t)(row - m) * 16 + li] = plus ? u[1][t][v] : u[0][t][v];
        }
}

// Back rotation of a segment's tiles and their sum: wave per (segment, degree), Z -> W.
template <int RT, int KS>
__device__ __forceinline__ void pair_back(int n, const PairSeg &G, const PairTile *__restrict__ tiles,
                                          const double *__restrict__ delta, const double2 *__restrict__ tab,
                                          const double *__restrict__ Z, double *__restrict__ w) {
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const int part = li & 3;
    const bool im = part & 1;
    DFrag<RT, KS> D;
    D.load(delta + delta_off(n), lane);
    double op[2][KS], om[2][KS];  // this lane's part at +-m, summed over the tiles
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int i = 0; i < KS; ++i) op[a][i] = om[a][i] = 0.0;
    for (int ti = G.t_begin; ti < G.t_end; ++ti) {
        const PairTile T = tiles[ti];
        const int K = T.K;
        const double2 *ph = tab + T.off_tab + (int64_t)(li >> 2) * T.tabw;
        const double2 *th = ph + T.NL + 1;
        const double *z = Z + T.off_z + (int64_t)yrow(n, 0, K) * 16;
        double vp[2][4 * RT], vm[2][4 * RT];
        rotate<RT, KS>(n, D, th, lane,
                       [&](int b, int c, double &p, double &q) {
                           const int k = b + 2 * c;
                           if (k > n || k > K) {
                               p = q = 0.0;
                               return;
                           }
                           const double sr = (c & 1) ? -1.0 : 1.0;
                           double up, um;
                           if (b == 0) {  // i^{+-k} = (-1)^c
                               up = sr * z[k * 16 + li];
                               um = sr * z[-k * 16 + li];
                           } else {       // +-i (-1)^c: the other part
                               const double f = im ? sr : -sr;
                               up = f * z[k * 16 + (li ^ 1)];
                               um = -f * z[-k * 16 + (li ^ 1)];
                           }
                           p = k == 0 ? up : up + um;
                           q = k == 0 ? 0.0 : up - um;
                       },
                       vp, vm);
        const double sg = im ? -1.0 : 1.0;
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int i = 0; i < KS; ++i) {
                const int m = a + 2 * (4 * i + lk);
                const double2 f = ph[m < n ? m : n];
                const double x = vp[a][i], y = vm[a][i];
                const double xo = __shfl_xor(x, 1, 64), yo = __shfl_xor(y, 1, 64);
                // (-1)^m conj(f) at +m, (-1)^m f at -m
                const double sm = a ? -1.0 : 1.0;
                op[a][i] += sm * (f.x * x + sg * f.y * xo);
                om[a][i] += sm * (f.x * y - sg * f.y * yo);
            }
    }
    // sum of the four slots, then a = (w_+ + w_-)/2, b = (w_+ - w_-)/2
    const int nent = G.Lt * (G.Lt + 2);
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int i = 0; i < KS; ++i) {
            const int m = a + 2 * (4 * i + lk);
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                double x = d == 0 ? op[a][i] : om[a][i];
                x += __shfl_xor(x, 4, 64);
                x += __shfl_xor(x, 8, 64);
                const double o = __shfl_xor(x, 2, 64);
                const double r = part < 2 ? 0.5 * (x + o) : 0.5 * (o - x);
                if (li >= 4 || m > n || (d == 1 && m == 0)) continue;
                const int e = n * n - 1 + n + (d == 0 ? m : -m) + (part < 2 ? 0 : nent);
                w[2 * (int64_t)e + (part & 1)] = r;
            }
        }
}

template <int RT, int KSM>
__global__ __launch_bounds__(256) void k_pair_back(const PairTile *__restrict__ tiles,
                                                   const PairSeg *__restrict__ segs, int s0, int nsegs, int n0,
                                                   const double *__restrict__ delta, const double2 *__restrict__ tab,
                                                   const double *__restrict__ Z, int64_t z_stride,
                                                   double2 *__restrict__ W, int64_t w_stride) {
    const int si = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    if (si >= nsegs) return;
    const PairSeg G = segs[s0 + si];
    const int n = n0 + blockIdx.y;
    if (n > G.Lt) return;
    const double *z = Z + blockIdx.z * z_stride;
    double *w = (double *)(W + blockIdx.z * w_stride + G.off_w);
    switch (n >> 3) {
        case 4 * (RT - 1): pair_back<RT, 4 * RT - 3>(n, G, tiles, delta, tab, z, w); break;
        case 4 * (RT - 1) + 1: pair_back<RT, 4 * RT - 2>(n, G, tiles, delta, tab, z, w); break;
        case 4 * (RT - 1) + 2:
            if constexpr (KSM > 4 * RT - 2) pair_back<RT, 4 * RT - 1>(n, G, tiles, delta, tab, z, w);
            break;
        default:
            if constexpr (KSM > 4 * RT - 1) pair_back<RT, 4 * RT>(n, G, tiles, delta, tab, z, w);
    }
}

// dst += the partial sums of a target's segments, in their order.
__global__ __launch_bounds__(256) void k_pair_reduce(const PairTarget *__restrict__ targets,
                                                     const PairSeg *__restrict__ segs, int g0,
                                                     const double2 *__restrict__ W, int64_t w_stride,
                                                     double2 *__restrict__ dst, int64_t dst_stride) {
    const PairTarget G = targets[g0 + blockIdx.x];
    const int nent = 2 * G.Lt * (G.Lt + 2);
    const double2 *w = W + blockIdx.z * w_stride;
    double2 *d = dst + blockIdx.z * dst_stride + G.dst;
    const int64_t o0 = segs[G.s_begin].off_w;  // the segments of a target lie one after another
    for (int e = blockIdx.y * 256 + threadIdx.x; e < nent; e += 256 * gridDim.y) {
        double2 a = d[e];
        for (int s = 0; s < G.s_end - G.s_begin; ++s) {
            const double2 v = w[o0 + (int64_t)s * nent + e];
            a.x += v.x;
            a.y += v.y;
        }
        d[e] = a;
    }
}

static void zero_doubles(double *p, size_t n, hipStream_t s) {
    launch_zero((double2 *)p, (int64_t)(n / 2), s);  // both kinds hold a multiple of 64 doubles
}

void launch_pair_delta(int NL, double *delta, size_t n_delta, hipStream_t s) {
    zero_doubles(delta, n_delta, s);
    hipLaunchKernelGGL(k_pair_delta, dim3(NL + 1), dim3(64), 0, s, NL, delta);
}

void launch_pair_quad(int NL, int Q, const double *mu, double *mats, size_t n_mats, hipStream_t s) {
    zero_doubles(mats, n_mats, s);
    hipLaunchKernelGGL(k_pair_quad, dim3(NL + 1, 2), dim3(Q), 0, s, NL, Q, mu, mats);
}

void launch_pair_tables(const PairTile *tiles, const PairSlot *slots, int t0, int ntiles, int max_P, const double *quad,
                        double2 *tab, hipStream_t s) {
    if (ntiles <= 0) return;
    hipLaunchKernelGGL(k_pair_tables, dim3(4 * ntiles), dim3(64), sizeof(double2) * (size_t)(max_P + 2), s, tiles,
                       slots, t0, quad, tab);
}

// Calls launch(KSM, first degree, degrees) for the degrees up to 31: by range from 512 waves a
// degree, else at once (small calls are bound by launches).  Near field of 2500 spheres,
// orders up to 23, forward and backward: 302 + 451 us a chunk in one launch with room for four
// steps, 270 + 333 with three for the backward one, 270 + 302 by range; a range of its own for
// degrees up to 7 gave nothing more.
template <typename F> static void by_steps(int64_t waves, int max_n, F launch) {
    const int lo = std::min(max_n, 31);
    if (waves < 512) {
        launch(std::max(2, (lo >> 3) + 1), 1, lo);
        return;
    }
    launch(2, 1, std::min(lo, 15));
    if (lo > 15) launch(3, 16, std::min(lo, 23) - 15);
    if (lo > 23) launch(4, 24, lo - 23);
}

void launch_pair_fwd(const PairTile *tiles, const PairSlot *slots, int t0, int ntiles, int max_Ls, const double *delta,
                     const double2 *tab, const double2 *src, int64_t src_stride, double *Y, int64_t y_stride, int nrhs,
                     hipStream_t s) {
    if (ntiles <= 0) return;
    by_steps((int64_t)ntiles * nrhs, max_Ls, [&](int ksm, int n0, int cnt) {
        auto k = ksm == 2 ? k_pair_fwd<1, 2> : ksm == 3 ? k_pair_fwd<1, 3> : k_pair_fwd<1, 4>;
        hipLaunchKernelGGL(k, dim3((ntiles + 3) / 4, cnt, nrhs), dim3(256), 0, s, tiles, slots, t0, ntiles, n0, delta,
                           tab, src, src_stride, Y, y_stride);
    });
    if (max_Ls > 31)
        hipLaunchKernelGGL((k_pair_fwd<2, 8>), dim3((ntiles + 3) / 4, max_Ls - 31, nrhs), dim3(256), 0, s, tiles, slots,
                           t0, ntiles, 32, delta, tab, src, src_stride, Y, y_stride);
}
void launch_pair_axial(const PairTile *tiles, const PairSlot *slots, const PairGroup *groups, int ngroups,
                       const int32_t *order, int waves, int max_K, int max_L, int NL, const double *quad,
                       const double2 *tab, const double2 *wax, const double *Y, int64_t y_stride, double *Z,
                       int64_t z_stride, int nrhs, hipStream_t s) {
    if (ngroups <= 0) return;
    const dim3 grid(ngroups, max_K + 1, nrhs);
#define IFS_PAIR_AXIAL(UT, KS)                                                                                      \
    hipLaunchKernelGGL((waves == 8 ? k_pair_axial<UT, KS, 8> : k_pair_axial<UT, KS, 4>), grid, dim3(64 * waves), 0, s,  \
                       tiles, slots, groups, order, NL, quad, tab, wax, Y, y_stride, Z, z_stride)
    if (max_L <= 16)
        IFS_PAIR_AXIAL(1, 4);
    else if (max_L <= 24)
        IFS_PAIR_AXIAL(2, 6);
    else if (max_L <= 32)
        IFS_PAIR_AXIAL(2, 8);
    else
        IFS_PAIR_AXIAL(4, 16);
#undef IFS_PAIR_AXIAL
}

void launch_pair_back(const PairTile *tiles, const PairSeg *segs, int s0, int nsegs, int max_Lt, const double *delta,
                      const double2 *tab, const double *Z, int64_t z_stride, double2 *W, int64_t w_stride, int nrhs,
                      hipStream_t s) {
    if (nsegs <= 0) return;
    by_steps((int64_t)nsegs * nrhs, max_Lt, [&](int ksm, int n0, int cnt) {
        auto k = ksm == 2 ? k_pair_back<1, 2> : ksm == 3 ? k_pair_back<1, 3> : k_pair_back<1, 4>;
        hipLaunchKernelGGL(k, dim3((nsegs + 3) / 4, cnt, nrhs), dim3(256), 0, s, tiles, segs, s0, nsegs, n0, delta, tab,
                           Z, z_stride, W, w_stride);
    });
    if (max_Lt > 31)
        hipLaunchKernelGGL((k_pair_back<2, 8>), dim3((nsegs + 3) / 4, max_Lt - 31, nrhs), dim3(256), 0, s, tiles, segs,
                           s0, nsegs, 32, delta, tab, Z, z_stride, W, w_stride);
}
void launch_pair_reduce(const PairTarget *targets, const PairSeg *segs, int g0, int ntargets, int max_Lt,
                        const double2 *W, int64_t w_stride, double2 *dst, int64_t dst_stride, int nrhs, hipStream_t s) {
    if (ntargets <= 0) return;
    const int yb = (2 * max_Lt * (max_Lt + 2) + 255) / 256;
    hipLaunchKernelGGL(k_pair_reduce, dim3(ntargets, yb, nrhs), dim3(256), 0, s, targets, segs, g0, W, w_stride, dst,
                       dst_stride);
}

}  // namespace ifs
