// Box-to-box translations (M2L) of one octree level in the plane-wave basis.
// Host declarations of ifs_pw.hip / ifs_pw.cpp.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <array>
#include <vector>

#include "ifs_engine.h"

namespace ifs {

constexpr int kPwMaxN = 4096;  // longest azimuthal transform (64 KiB of LDS)

// One source box seen from a parent: its children in `mask` receive it.
struct PwSource {
    int32_t box;   // source box of the level
    int32_t r;     // ((rx + 2) * 6 + ry + 2) * 6 + rz + 2: source minus 2 * parent, -2..3 each
    int32_t mask;  // children (bit c = 4 cx + 2 cy + cz) whose offset r - c is translated here
    int32_t pad_;
};
struct PwParent {
    int32_t child[8];  // box of each octant, -1: empty
    int32_t beg, end;  // sources
};
// How the offset of (source position, child) reads the canonical tables.
struct PwMap {
    int32_t table;   // canonical offset
    int32_t flip;    // 1: polar angle mirrored
    int32_t sign;    // +1, -1: azimuth i -> sign * i + shift * N / 4
    int32_t shift;
};
struct PwMaps {
    PwMap child[8];
};
// Azimuthal transform of one length.
struct PwFft {
    int32_t N, npass;
    int32_t radix[12];
    int32_t tw, perm;  // offsets of the twiddles (complex) and of the digit-reversal table
};

struct PwLevel {
    int L = 0, nb = 0;
    int64_t off = 0;          // pool offset of the first box (complex)
    double k = 0.0, edge = 0.0;
    int Q2 = 0;               // nodes per hemisphere; position t < Q2: node t, t >= Q2: its mirror
    std::vector<int> N, mF;   // per node: azimuths, largest |m| kept
    std::vector<int> jlo;     // per |m|: first node with mF >= |m|
    std::vector<PwSource> src;
    std::vector<PwParent> par;
    std::vector<PwMaps> map;  // [216]
    std::vector<std::array<int, 3>> canon;
    std::vector<PwFft> fft;   // distinct lengths
    std::vector<int> fft_of;  // per node
    int64_t ncols = 0;        // translations
    DevBuf d_mu, d_N, d_mF, d_jlo, d_src, d_par, d_map, d_fft, d_fftof, d_tw, d_perm, d_gpre, d_hank, d_canon;
    DevBuf own_U, own_T, own_T32;  // T in FP64, and in FP32 for mixed products
    bool kept = false, ready = false;
    bool t_ready[2] = {false, false};
    bool no_t32 = false;      // the budget or the device has no room for the FP32 copy: mixed products read T
    int64_t SN = 0;           // azimuths of all positions
    struct Chunk {
        int j0, R2;           // nodes [j0, j0 + R2) and their mirrors
        int64_t sn;           // azimuths of the chunk's rows
        int maxN;
        double f_gemm, f_fft; // algorithmic flops of one direction, per box (pw_row_flops)
    };
    std::vector<Chunk> chunks;
    DevBuf d_cpre;            // per chunk: prefix of N over its 2 R2 rows, chunk after chunk
    std::vector<int64_t> cpre_at;
    int plan_nrhs = 0;        // right-hand sides the plan was cut for, 0: no valid plan
    WsNeed ws;
    int64_t n_x = 0, n_g = 0, n_f = 0, n_u = 0, n_t = 0;  // complex (u: doubles)
    bool active() const { return ncols > 0; }
};

// Last degree P of h1 that the plane waves carry for offsets of squared length o2 (box
// edges), at most 2 L.  Beyond t = k |d| |h1_p| grows, and its size is rounding noise in
// every degree; at (P - t)/(t/2)^{1/3} = 2.5 it has grown 16 to 27 times.
int pw_terms(double k, double edge, int o2, int L);
// Whether the plane waves take the offset: the degrees P + 1 - L .. L of the remaining
// terms cost a class product 1 - (n0/L)^3 of the rotations of a whole one, so not when
// n0 < L / 2 (7/8 would remain).
inline bool pw_takes(int P, int L) { return P >= 2 * L || P + 1 - L >= (L + 1) / 2; }
// Whether the level is worth it (rule and figures at the definition), given its
// translations by plane waves.
bool pw_worth(int L, int nb, int64_t cols);
// The grid of a level: 2 Q2 nodes, azimuths for fields of order L and `order` under factors
// whose azimuthal orders fall like J_m(tdeg sin(theta)), at most tcap.
int pw_grid(ifs_ctx *c, PwLevel &P, int Q2, double tdeg, int tcap, int order);
// The longest azimuthal transform of such a grid (that of a row at the equator).
int pw_max_azimuths(int L, double tdeg, int tcap, int order);
// parents: for every parent box its children and sources; called once per level.
int pw_build(ifs_ctx *c, PwLevel &P, int isg);
int pw_plan(ifs_ctx *c, PwLevel &P, int nrhs);  // leaves ws.s as it is
// Right-hand sides whose samples the workspace holds at once.  A level is planned for that many;
// the last, smaller group of a product runs on the same plan.
int pw_group(ifs_ctx *c, const PwLevel &P, int nrhs);
// The plan for nrhs right-hand sides (waits for the stream where it is cut anew), its workspaces and,
// for the first mixed product, the FP32 tables' room; pw_run asks for them itself.
int pw_prepare(ifs_ctx *c, PwLevel &P, int nrhs, int prec);
int pw_run(ifs_ctx *c, PwLevel &P, const double2 *C, double2 *D, int nrhs, int64_t stride, int prec);
bool pw_fits(size_t ws_budget, int L, int nb, int nrhs);
// Device bytes of a level on such a grid (pw_grid), counted without planning it: U, T of one canonical
// offset, and the workspaces of all rows in one chunk.
struct PwSize {
    double U = 0.0, T = 0.0, y = 0.0, z = 0.0;
    double samples = 0.0, box_flops = 0.0;  // of one box: azimuths of all rows; synthesis, analysis, transforms
};
PwSize pw_size(int L, int nbr, int Q2, double tdeg, int tcap, int order);
// Algorithmic flops of one product: the two GEMMs (8 Q degrees^2 each way per box), the
// azimuthal transforms (5 N log2 N), 16 per sample and translation.
double pw_flops(const PwLevel &P);
// One direction of one node and its mirror, per box: the products with U (complex by real, two
// helicities), and the azimuthal transforms.
void pw_row_flops(int L, int mF, int N, double &gemm, double &fft);
uint64_t pw_sig(const PwLevel &P);

// -- kernels --------------------------------------------------------------------
// sum_{q=1}^{j} (L - q + 1), and the degrees of order m
__host__ __device__ inline int64_t pw_sum(int j, int L) { return (int64_t)j * L - (int64_t)j * (j - 1) / 2; }
__host__ __device__ inline int pw_cn(int m, int L) {
    const int q = m < 0 ? -m : m;
    return L - (q < 1 ? 1 : q) + 1;
}
// degrees of orders 0..m-1 (rows of U before order m)
__host__ __device__ inline int64_t pw_ucnt(int m, int L) { return m < 1 ? 0 : L + pw_sum(m - 1, L); }
// degrees of orders -L..m-1 (rows of X before order m, per helicity)
__host__ __device__ inline int64_t pw_xcnt(int m, int L) {
    return m <= 0 ? pw_sum(L, L) - pw_sum(-m, L) : pw_sum(L, L) + L + pw_sum(m - 1, L);
}

struct PwArg {
    int L, nbr;            // order; boxes x right-hand sides
    int Q2, j0, R2;        // nodes per hemisphere, the chunk's first node and its count
    int a0, a1;            // table positions of the chunk's rows: a0 + lr, a1 + lr - R2
    int64_t ustr;          // positions per row of U
    const double *U;
    const int32_t *jlo, *mF, *N, *fftof;
    const PwFft *fft;
    const double2 *tw;
    const int32_t *perm;
    const int64_t *cpre;   // prefix of N over the chunk's rows
    const int64_t *tpre;   // prefix of N over table positions
    int64_t tsn;           // azimuths per canonical table
    const double2 *T;
    const float2 *T32;     // mixed precision: T rounded to FP32 (T unused)
    double2 *X, *Xd, *G, *F, *H;
};
PwArg pw_arg(ifs_ctx *c, const PwLevel &P, int nrhs);
void launch_pw_utable(int L, int Q2, int j0, int R2, int a0, int a1, int64_t ustr, const double *mu, double *U,
                      hipStream_t s);
// terms: last p of every table; c_p = 0 beyond it
void launch_pw_hankel(int ncanon, int P, const double *t, const int32_t *terms, double2 *h, hipStream_t s);
// canon: per table the direction (3) and t; tables at positions a0 + lr / a1 + lr - R2
void launch_pw_ttable(int ncanon, int P, int Q2, int j0, int R2, int a0, int a1, int maxN, const double *mu,
                      const double *canon, const int32_t *N, const int64_t *tpre, int64_t tsn, const double2 *h,
                      double2 *T, float2 *T32, hipStream_t s);
void launch_pw_pack(const PwArg &a, int nb, int64_t off, const double2 *C, int64_t stride, hipStream_t s);
void launch_pw_synth(const PwArg &a, hipStream_t s);
void launch_pw_fft(const PwArg &a, int inverse, int maxN, hipStream_t s);
void launch_pw_m2l(const PwArg &a, const PwParent *par, int npar, const PwSource *src, const PwMaps *map, int nb,
                   int nrhs, int maxN, hipStream_t s);
void launch_pw_anal(const PwArg &a, int accumulate, hipStream_t s);
void launch_pw_unpack(const PwArg &a, int nb, int64_t off, double2 *D, int64_t stride, hipStream_t s);

}  // namespace ifs
