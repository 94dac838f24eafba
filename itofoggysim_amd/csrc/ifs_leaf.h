// Sphere <-> leaf box translations (P2M, L2P) through samples of the box's field.
// Host declarations of ifs_leaf.hip / ifs_leaf.cpp.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "ifs_pw.h"

namespace ifs {

struct LeafSphere {
    int64_t off;   // complex offset of the sphere's expansion (a-part)
    int32_t N;     // order
    int32_t box;
    double v[3];   // exponent of the plane wave s: k * v . s
};

struct Leaf {
    PwLevel g;                     // leaf boxes and their grid (no translation tables)
    int Nmax = 0;
    std::vector<LeafSphere> up, down;   // P2M sources, L2P targets, both by box
    std::vector<int32_t> first;         // per box: first of its P2M sources (nb + 1)
    DevBuf d_up, d_down, d_first, d_us; // d_us: U of the sphere orders, [position][n (n+1)/2 + m]
    int64_t gcap = 0;                   // spheres whose row coefficients the workspace holds
    bool active() const { return g.nb > 0; }
};

// Largest sphere order and exponent of the translations.
struct LeafReach {
    int order = 0;
    double t = 0.0;
    void add(int N, double exponent) {
        order = N > order ? N : order;
        t = exponent > t ? exponent : t;
    }
    int deg() const;          // degree of the factor: (2p+1) j_p(t) vanishes beyond
    int nodes(int L) const;   // Q: 2 Q nodes integrate degree 4 Q - 1 >= L + order + deg
};
LeafReach leaf_reach(const std::vector<Task> &p2m, const std::vector<Task> &l2p);
// Whether the leaf level's spheres go this way (rule and figures at the definition).
bool leaf_worth(size_t ws_budget, const LeafReach &R, int L, int nb, int ns);
// p2m, l2p: the translations; off: pool offset of the first leaf box
int leaf_build(ifs_ctx *c, Leaf &F, const std::vector<Task> &p2m, const std::vector<Task> &l2p, int L, int nb,
               int64_t off);
// As pw_prepare.
int leaf_prepare(ifs_ctx *c, Leaf &F, int nrhs);
int leaf_p2m(ifs_ctx *c, Leaf &F, const double2 *xh, double2 *C, int nrhs, int64_t ldx, int64_t ldC);
int leaf_l2p(ifs_ctx *c, Leaf &F, const double2 *D, double2 *acc, int nrhs, int64_t ldD, int64_t ldacc);
uint64_t leaf_sig(const Leaf &F);

// Dynamic LDS of a block: the row sums of two spheres (P2M); a quarter of a row's azimuths in four
// classes and both helicities, and partial sums (L2P).
inline size_t leaf_p2m_lds(int Nmax) { return 16 * 4 * (size_t)(2 * Nmax + 1); }
inline size_t leaf_l2p_lds(int maxN) { return 16 * (8 * (size_t)(maxN / 4) + 128); }

// -- kernels --------------------------------------------------------------------
struct LeafArg {
    PwArg p;
    const double *mu;          // nodes, weights
    const double *us;          // U of the sphere orders
    int ucols;                 // entries per position
    int nb, Nmax;
};
void launch_leaf_utable(int Nmax, int Q2, int ucols, const double *mu, double *us, hipStream_t s);
// spheres s0 .. s0 + ns - 1: row sums into g, samples written or added to H
void launch_leaf_p2m(const LeafArg &a, const LeafSphere *sph, const int32_t *first, int s0, int ns, const double2 *xh,
                     int64_t ldx, int nrhs, int maxN, double2 *g, int accumulate, hipStream_t s);
// rows of the chunk -> coefficients of every order: g[(sphere - s0)][rhs][position][2][2 Nmax + 1]
void launch_leaf_l2p(const LeafArg &a, const LeafSphere *sph, int s0, int ns, int nrhs, int maxN, double2 *g,
                     hipStream_t s);
// acc += sum over all positions
void launch_leaf_sum(const LeafArg &a, const LeafSphere *sph, int s0, int ns, int nrhs, const double2 *g, double2 *acc,
                     int64_t ldacc, hipStream_t s);

}  // namespace ifs
