// Sphere-pair translations (direct plan, near field) with matrices shared by all pairs.
// Host declarations of ifs_pair.hip / ifs_pair.cpp.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <set>
#include <vector>

#include "ifs_engine.h"

namespace ifs {

// Largest order the pair kernels hold (two 16-row tiles of one parity).
constexpr int kPairMaxL = 63;

// Four translations of one target, advanced together as the 16 real columns of a
// matrix-core tile: column 4 s + p is part p of slot s (Re, Im of x_+, then of x_-).
struct PairTile {
    int64_t off_y;    // rotated sources: rows_size(Ls, K) rows of 16 doubles
    int64_t off_z;    // shifted: rows_size(Lt, K) rows of 16 doubles
    int64_t off_tab;  // complex: 4 slots of tabw entries, each e^{im(phi - pi/2)}, e^{-ij theta}, w_q T(mu_q)
    int32_t Ls, Lt, K;  // largest source order of the slots, target order, min
    int32_t NL;       // max(Ls, Lt): entries of the two phase rows less one
    int32_t Q;        // quadrature nodes (a multiple of 16); 0: coaxial tables (close pairs)
    int32_t tabw;     // 2 (NL + 1) + Q
    int64_t off_q;    // offset (doubles) of the quadrature matrices of this Q
    int64_t off_mu;   // ... and of its nodes, then weights
};
struct PairSlot {
    int64_t src;      // complex offset of the source expansion; -1: empty slot
    int64_t off_ax;   // complex offset of the coaxial table (close pairs)
    double t, cth, phi;
    int32_t Ls, K;
};
// Consecutive tiles of one target summed by one wave, and the partial sum it writes.
struct PairSeg {
    int64_t off_w;    // complex offset of the partial sum, 2 Lt (Lt + 2) entries
    int32_t Lt, t_begin, t_end, pad_;
};
// Tiles of one node set (positions first .. of the order list) shifted by one block.
struct PairGroup {
    int32_t first, count, Q, Ls, Lt, K;  // largest orders of its tiles
    int64_t off_q;
};
struct PairTarget {
    int64_t dst;      // complex offset of the target expansion
    int32_t Lt, s_begin, s_end, pad_;
};

struct PairBatch {
    struct Chunk {
        int t0 = 0, t1 = 0, s0 = 0, s1 = 0, g0 = 0, g1 = 0, c0 = 0, c1 = 0;  // tiles, segments, targets, close tasks
        int a0 = 0, a1 = 0, waves = 4;  // groups, tiles of a group
        int64_t n_y = 0, n_z = 0, n_w = 0, n_tab = 0, n_ax = 0, n_s = 0;
        int max_Ls = 0, max_Lt = 0, max_K = 0, maxK_close = 0, max_nmax = 0, max_P = 0;
        double f_fwd = 0.0, f_ax = 0.0, f_back = 0.0;
    };
    std::vector<PairTile> tiles;
    std::vector<PairSlot> slots;
    std::vector<PairSeg> segs;
    std::vector<PairTarget> targets;
    std::vector<PairGroup> groups;
    std::vector<int32_t> order;  // tiles of a chunk by node set
    std::vector<Task> close;  // coaxial tables by the degree recurrence
    std::vector<Chunk> chunks;
    DevBuf d_tiles, d_slots, d_segs, d_targets, d_close, d_groups, d_order;
    DevBuf d_delta, d_quad;   // shared matrices
    DevBuf own_tab, own_ax;   // tables kept across matvecs
    bool kept = false, ready = false;
    // Offsets of the spheres' sums, where the caller can take partial sums: with all tiles in
    // one chunk no pass adds them, and d_parts holds those of every sphere.
    std::vector<int64_t> rows;
    DevBuf d_parts;
    int64_t n_y = 0, n_z = 0, n_w = 0, n_s = 0;  // largest chunk, per right-hand side (n_s: for all)
    WsNeed ws;                // tables that are not kept
    int NL = 0;               // orders of the shared matrices
    std::vector<Task> tasks;  // the translations, sorted by target
    const char *pn[4] = {"gen_tables", "rot_fwd", "axial_apply", "rot_back"};
    bool active() const { return !tasks.empty(); }
};

// Whether the pair kernels take these translations (outgoing -> regular, orders <= kPairMaxL).
bool pair_takes(const std::vector<Task> &tasks);
// Takes the tasks over and plans them, for any number of right-hand sides.
int pair_finalize(ifs_ctx *c, PairBatch &B, std::vector<Task> &tasks, const char *name);
// Whether a product leaves partial sums in ws_s to its caller (d_parts) and adds nothing to dst_pool.
bool pair_parts(const ifs_ctx *c, const PairBatch &B, int nrhs);
// Device bytes and algorithmic flops of a plan, counted target by target without planning it
// (admission of served requests).
struct PairSize {
    double tables = 0.0, work = 0.0;  // kept tables; Y, Z and partial sums of one right-hand side
    double sect = 0.0, lists = 0.0;   // workspace of the close pairs' tables; tiles, slots and the rest
    double flops = 0.0;               // 21 L^3 a pair, L the larger order
    int NL = 0;
    std::set<int> nodes;
    double shared() const;            // d(pi/2) and the node sets
};
// Adds one target's translations `weight` times.
void pair_size(const std::vector<Task> &of_target, double weight, PairSize &S);
// Largest workspace of the rotated and shifted columns, whatever the budget.
double pair_work_cap();
// The workspaces of a product of nrhs right-hand sides; pair_run asks for them itself.
int pair_prepare(ifs_ctx *c, const PairBatch &B, int nrhs);
int pair_run(ifs_ctx *c, PairBatch &B, const double2 *src_pool, double2 *dst_pool, int nrhs, int64_t src_stride,
             int64_t dst_stride);
uint64_t pair_sig(const PairBatch &B);

// -- kernels (ifs_pair.hip) -----------------------------------------------------
__host__ __device__ inline int pair_rt(int n) { return n < 32 ? 1 : 2; }
__host__ __device__ inline int pair_ks(int n) { return (n / 2 + 4) / 4; }
// doubles before degree n: sum_{i=1}^{n-1} 4 rt ks 64
inline int64_t pair_delta_off_host(int n) {
    int64_t s = 0;
    for (int i = 1; i < n; ++i) s += 256LL * pair_rt(i) * pair_ks(i);
    return s;
}
// The shared matrices: d^n(pi/2) (n_delta doubles in all), and those of one node set.
void launch_pair_delta(int NL, double *delta, size_t n_delta, hipStream_t s);
void launch_pair_quad(int NL, int Q, const double *mu, double *mats, size_t n_mats, hipStream_t s);
void launch_pair_tables(const PairTile *tiles, const PairSlot *slots, int t0, int ntiles, int max_P, const double *quad,
                        double2 *tab, hipStream_t s);
void launch_pair_fwd(const PairTile *tiles, const PairSlot *slots, int t0, int ntiles, int max_Ls, const double *delta,
                     const double2 *tab, const double2 *src, int64_t src_stride, double *Y, int64_t y_stride, int nrhs,
                     hipStream_t s);
void launch_pair_axial(const PairTile *tiles, const PairSlot *slots, const PairGroup *groups, int ngroups,
                       const int32_t *order, int waves, int max_K, int max_L, int NL, const double *quad,
                       const double2 *tab, const double2 *wax, const double *Y, int64_t y_stride, double *Z,
                       int64_t z_stride, int nrhs, hipStream_t s);
void launch_pair_back(const PairTile *tiles, const PairSeg *segs, int s0, int nsegs, int max_Lt, const double *delta,
                      const double2 *tab, const double *Z, int64_t z_stride, double2 *W, int64_t w_stride, int nrhs,
                      hipStream_t s);
void launch_pair_reduce(const PairTarget *targets, const PairSeg *segs, int g0, int ntargets, int max_Lt,
                        const double2 *W, int64_t w_stride, double2 *dst, int64_t dst_stride, int nrhs, hipStream_t s);

}  // namespace ifs
