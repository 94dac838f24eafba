// Plan and launch order of the sphere-pair translations (kernels: ifs_pair.hip).
#include "ifs_pair.h"

#include <algorithm>
#include <cmath>
#include <map>

namespace ifs {

namespace {

// Columns of one right-hand side rotated and shifted at once, and of all that run together.
constexpr size_t kPairChunk = (size_t)1 << 30, kPairWork = 4 * kPairChunk;

// Largest growth of |h1_p(t)| up to the last order P = Ls + Lt that the quadrature may
// carry: |h1_P| / |h1_0| follows exp(2/3 z^{3/2}) in z = (P - t) / (t/2)^{1/3}; at z = 2.5
// it is 16 to 27 for every P from 3 to 126 (evaluated), so the quadrature rounds within
// a few 1e-15 of the largest entry.  Closer pairs take tables from the degree recurrence.
bool is_close(const Task &T) {
    const double P = (double)(T.Ls + T.Lt);
    return P - T.t > 2.5 * std::cbrt(0.5 * T.t);
}

// Doubles of one node set's two operand-ordered matrices.
size_t quad_size(int L, int Q) {
    const size_t QT = Q / 16, S1 = (L + 3) / 4, UT = (L + 15) / 16;
    return (size_t)(L + 1) * 2 * QT * 64 * (S1 + 4 * UT);
}

int upload(DevBuf &d, const void *h, size_t bytes) {
    int rc = d.alloc(std::max<size_t>(bytes, 16));
    if (rc) return rc;
    if (bytes && hipMemcpy(d.p, h, bytes, hipMemcpyHostToDevice) != hipSuccess) return IFS_E_HIP;
    return IFS_OK;
}

// Tiles of at most four translations of one target (sources by order, close pairs apart).
void build_tiles(PairBatch &B, std::map<int, int64_t> &quads) {
    std::vector<Task> far, close;
    for (size_t i = 0; i < B.tasks.size();) {
        size_t j = i;
        far.clear();
        close.clear();
        for (; j < B.tasks.size() && B.tasks[j].dst == B.tasks[i].dst; ++j)
            (is_close(B.tasks[j]) ? close : far).push_back(B.tasks[j]);
        for (auto *v : {&far, &close}) {
            std::stable_sort(v->begin(), v->end(), [](const Task &a, const Task &b) { return a.Ls < b.Ls; });
            for (size_t a = 0; a < v->size(); a += 4) {
                const size_t n = std::min<size_t>(4, v->size() - a);
                PairTile T{};
                T.Ls = (*v)[a + n - 1].Ls;
                T.Lt = (*v)[a].Lt;
                T.K = std::min(T.Ls, T.Lt);
                T.NL = std::max(T.Ls, T.Lt);
                T.Q = v == &far ? (T.Ls + T.Lt + 1 + 15) / 16 * 16 : 0;
                T.tabw = 2 * (T.NL + 1) + T.Q;
                if (T.Q) quads[T.Q] = 0;
                for (size_t s = 0; s < 4; ++s) {
                    const Task &K = (*v)[a + std::min(s, n - 1)];
                    PairSlot S{};
                    S.src = s < n ? K.src : -1;
                    S.t = K.t;
                    S.cth = K.cth;
                    S.phi = K.phi;
                    S.Ls = K.Ls;
                    S.K = K.K;
                    B.slots.push_back(S);
                }
                B.tiles.push_back(T);
            }
        }
        i = j;
    }
}

WsNeed pair_need(const PairBatch &B, int nrhs) {
    WsNeed w = B.ws;
    w.y = 8 * (size_t)B.n_y * nrhs;
    w.z = 8 * (size_t)B.n_z * nrhs;
    w.s = 16 * (size_t)std::max<int64_t>(B.n_w * nrhs, B.n_s);
    return w;
}

// Chunks, segments and per-chunk target lists; workspace offsets.  Cut for one right-hand
// side: products of several run as many together as the largest chunk leaves room for.
int pair_plan(ifs_ctx *c, PairBatch &B) {
    B.chunks.clear();
    B.segs.clear();
    B.targets.clear();
    B.close.clear();
    const size_t budget = std::max<size_t>(std::min(c->ws_budget, kPairChunk), 1);
    // first tile of every target
    std::vector<size_t> first;
    std::vector<int64_t> dst;
    {
        size_t tile = 0;
        for (size_t i = 0; i < B.tasks.size();) {
            size_t j = i, nf = 0, nc = 0;
            for (; j < B.tasks.size() && B.tasks[j].dst == B.tasks[i].dst; ++j) ++(is_close(B.tasks[j]) ? nc : nf);
            first.push_back(tile);
            dst.push_back(B.tasks[i].dst);
            tile += (nf + 3) / 4 + (nc + 3) / 4;
            i = j;
        }
        first.push_back(tile);
    }
    // algorithmic flops of a folded rotation of order L with |k| <= K
    std::vector<double> rot((size_t)(kPairMaxL + 1) * (kPairMaxL + 1), 0.0);
    for (int L = 1; L <= kPairMaxL; ++L)
        for (int K = 0; K <= L; ++K) {
            const double kk = std::min(L, K);
            const double below = L > 1 ? rot[(L - 1) * (kPairMaxL + 1) + std::min(K, L - 1)] : 0.0;
            rot[L * (kPairMaxL + 1) + K] = below + 8.0 * ((kk + 1.0) * (L + 1.0) + kk * L);
        }
    PairBatch::Chunk cur;
    size_t used = 0;
    int64_t tab = 0, ax = 0;  // running table offsets when the tables are kept
    auto close_chunk = [&]() {
        cur.t1 = (int)(B.segs.empty() ? 0 : B.segs.back().t_end);
        cur.s1 = (int)B.segs.size();
        cur.g1 = (int)B.targets.size();
        cur.c1 = (int)B.close.size();
        B.chunks.push_back(cur);
        PairBatch::Chunk n;
        n.t0 = cur.t1;
        n.s0 = cur.s1;
        n.g0 = cur.g1;
        n.c0 = cur.c1;
        cur = n;
        used = 0;
    };
    for (size_t g = 0; g + 1 < first.size(); ++g) {
        const int nt = (int)(first[g + 1] - first[g]);
        // tiles one wave sums: eight partial sums per target at most eight tiles long.  A
        // target's sum then does not depend on what else the plan holds.
        const int G = std::min(8, (nt + 7) / 8);
        bool open = false;
        for (size_t a = first[g]; a < first[g + 1]; a += G) {
            const size_t b = std::min(first[g + 1], a + G);
            size_t bytes = 0;
            for (size_t t = a; t < b; ++t) {
                const PairTile &T = B.tiles[t];
                bytes += 128 * (size_t)(rows_size(T.Ls, T.K) + rows_size(T.Lt, T.K));
                if (!B.kept) {
                    bytes += 64 * (size_t)T.tabw;
                    for (int s = 0; s < 4 && T.Q == 0; ++s)
                        bytes += 16 * (size_t)(ax_size(T.Lt, B.slots[4 * t + s].Ls, B.slots[4 * t + s].K) +
                                               sect_size(B.slots[4 * t + s].K, T.Lt + B.slots[4 * t + s].Ls + 2));
                }
            }
            bytes += 32 * (size_t)B.tiles[a].Lt * (B.tiles[a].Lt + 2);
            if (used && used + bytes > budget) {
                close_chunk();
                open = false;
            }
            used += bytes;
            const int Lt = B.tiles[a].Lt;
            if (!open) {
                B.targets.push_back({dst[g], Lt, (int)B.segs.size(), 0, 0});
                open = true;
            }
            B.segs.push_back({cur.n_w, Lt, (int)a, (int)b, 0});
            B.targets.back().s_end = (int)B.segs.size();
            cur.n_w += 2LL * Lt * (Lt + 2);
            for (size_t t = a; t < b; ++t) {
                PairTile &T = B.tiles[t];
                T.off_y = cur.n_y;
                T.off_z = cur.n_z;
                cur.n_y += 16 * rows_size(T.Ls, T.K);
                cur.n_z += 16 * rows_size(T.Lt, T.K);
                int64_t &nt_ = B.kept ? tab : cur.n_tab, &na_ = B.kept ? ax : cur.n_ax;
                T.off_tab = nt_;
                nt_ += 4LL * T.tabw;
                cur.max_Ls = std::max(cur.max_Ls, T.Ls);
                cur.max_Lt = std::max(cur.max_Lt, T.Lt);
                cur.max_K = std::max(cur.max_K, T.K);
                cur.max_P = std::max(cur.max_P, T.Ls + T.Lt);
                for (int s = 0; s < 4; ++s) {
                    PairSlot &S = B.slots[4 * t + s];
                    if (S.src < 0) continue;
                    cur.f_fwd += rot[S.Ls * (kPairMaxL + 1) + S.K];
                    cur.f_back += rot[T.Lt * (kPairMaxL + 1) + S.K];
                    cur.f_ax += 8.0 * (double)ax_size(T.Lt, S.Ls, S.K);
                    if (T.Q) continue;
                    Task K{};
                    K.t = S.t;
                    K.Ls = T.Lt;  // source and target change places (see the kernel)
                    K.Lt = S.Ls;
                    K.K = S.K;
                    K.kind = IFS_ZSEL_HANKEL1;
                    S.off_ax = K.off_ax = na_;
                    K.off_s = cur.n_s;
                    na_ += ax_size(T.Lt, S.Ls, S.K);
                    cur.n_s += sect_size(S.K, T.Lt + S.Ls + 2);
                    cur.maxK_close = std::max(cur.maxK_close, S.K);
                    cur.max_nmax = std::max(cur.max_nmax, T.Lt + S.Ls + 2);
                    B.close.push_back(K);
                }
            }
        }
    }
    if (cur.t0 < (int)B.tiles.size()) close_chunk();
    // tiles by node set, then by order, 8 to a block of the shift (4 where a chunk has few)
    B.groups.clear();
    B.order.clear();
    for (auto &ch : B.chunks) {
        // with twice the tiles a block reads the shift matrices half as often, at twice the tiles that
        // wait for its slowest: 1056 to 5775 tiles of orders up to 22 77 -> 66 to 381 -> 313 us with
        // eight, of orders up to 11 30 -> 31 to 131 -> 135; 110 tiles 20.5 -> 21.1 (with 420, orders up
        // to 22, eight would be the better already: 35.5 -> 30.7)
        ch.waves = ch.t1 - ch.t0 >= 1024 ? 8 : 4;
        std::vector<int32_t> o;
        for (int t = ch.t0; t < ch.t1; ++t) o.push_back(t);
        std::stable_sort(o.begin(), o.end(), [&](int a, int b) {
            const PairTile &x = B.tiles[a], &y = B.tiles[b];
            return x.Q != y.Q ? x.Q < y.Q : x.K < y.K;
        });
        ch.a0 = (int)B.groups.size();
        for (size_t i = 0; i < o.size();) {
            const PairTile &T = B.tiles[o[i]];
            PairGroup G{(int)(B.order.size() + i), 0, T.Q, 0, 0, 0, T.off_q};
            for (; i < o.size() && G.count < ch.waves && B.tiles[o[i]].Q == G.Q; ++i, ++G.count) {
                G.Ls = std::max(G.Ls, B.tiles[o[i]].Ls);
                G.Lt = std::max(G.Lt, B.tiles[o[i]].Lt);
                G.K = std::max(G.K, B.tiles[o[i]].K);
            }
            B.groups.push_back(G);
        }
        ch.a1 = (int)B.groups.size();
        B.order.insert(B.order.end(), o.begin(), o.end());
    }
    std::vector<SphereParts> parts;
    if (!B.rows.empty() && B.chunks.size() == 1) {
        std::map<int64_t, size_t> at;
        for (size_t j = 0; j < B.rows.size(); ++j) at[B.rows[j]] = j;
        parts.assign(B.rows.size(), SphereParts{0, 0, 0});
        for (const PairTarget &T : B.targets)
            parts[at[T.dst]] = SphereParts{B.segs[T.s_begin].off_w, T.s_end - T.s_begin, 0};
    }
    B.n_y = B.n_z = B.n_w = B.n_s = 0;
    int64_t mt = 0, ma = 0;
    for (auto &ch : B.chunks) {
        B.n_y = std::max(B.n_y, ch.n_y);
        B.n_z = std::max(B.n_z, ch.n_z);
        B.n_w = std::max(B.n_w, ch.n_w);
        B.n_s = std::max(B.n_s, ch.n_s);
        mt = std::max(mt, ch.n_tab);
        ma = std::max(ma, ch.n_ax);
    }
    int rc;
    B.ws.d = B.kept ? 0 : 16 * (size_t)mt;
    B.ws.ax = B.kept ? 0 : 16 * (size_t)ma;
    if ((rc = ws_reserve(c, pair_need(B, 1)))) return rc;
    if ((rc = upload(B.d_tiles, B.tiles.data(), sizeof(PairTile) * B.tiles.size())) ||
        (rc = upload(B.d_slots, B.slots.data(), sizeof(PairSlot) * B.slots.size())) ||
        (rc = upload(B.d_segs, B.segs.data(), sizeof(PairSeg) * B.segs.size())) ||
        (rc = upload(B.d_targets, B.targets.data(), sizeof(PairTarget) * B.targets.size())) ||
        (rc = upload(B.d_groups, B.groups.data(), sizeof(PairGroup) * B.groups.size())) ||
        (!parts.empty() && (rc = upload(B.d_parts, parts.data(), sizeof(SphereParts) * parts.size()))) ||
        (rc = upload(B.d_order, B.order.data(), 4 * B.order.size())) ||
        (rc = upload(B.d_close, B.close.data(), sizeof(Task) * B.close.size())))
        return rc;
    return IFS_OK;
}

// Right-hand sides run together: launches of one right-hand side each end in a last wave that
// is nearly empty (near field of 450 spheres with four: 3.44 ms in turn, 3.33 as chunks cut for
// all four in 1 GiB, 3.21 together).
int pair_group(const ifs_ctx *c, const PairBatch &B, int nrhs) {
    const size_t budget = std::min(c->ws_budget, kPairWork), tab = B.ws.d + B.ws.ax;
    const size_t one = 8 * (size_t)(B.n_y + B.n_z + 2 * B.n_w);
    const size_t g = budget > tab ? (budget - tab) / std::max<size_t>(one, 1) : 1;
    return (int)std::min<size_t>((size_t)nrhs, std::max<size_t>(g, 1));
}

}  // namespace

bool pair_takes(const std::vector<Task> &tasks) {
    for (auto &T : tasks)
        if (T.kind != IFS_ZSEL_HANKEL1 || T.Ls > kPairMaxL || T.Lt > kPairMaxL || !(T.t > 0.0)) return false;
    return !tasks.empty();
}

double pair_work_cap() { return (double)kPairWork; }

void pair_size(const std::vector<Task> &of_target, double weight, PairSize &S) {
    if (of_target.empty()) return;
    PairBatch B;
    B.tasks = of_target;
    std::map<int, int64_t> quads;
    build_tiles(B, quads);
    for (size_t t = 0; t < B.tiles.size(); ++t) {
        const PairTile &T = B.tiles[t];
        S.tables += weight * 64.0 * T.tabw;
        S.work += weight * 128.0 * (double)(rows_size(T.Ls, T.K) + rows_size(T.Lt, T.K));
        for (int s = 0; s < 4 && !T.Q; ++s) {
            const PairSlot &P = B.slots[4 * t + s];
            if (P.src < 0) continue;
            S.tables += weight * 16.0 * (double)ax_size(T.Lt, P.Ls, P.K);
            S.sect += weight * 16.0 * (double)sect_size(P.K, T.Lt + P.Ls + 2);
            S.lists += weight * sizeof(Task);
        }
    }
    // at most eight partial sums a target
    const double nt = (double)B.tiles.size(), L = of_target[0].Lt;
    S.work += weight * 32.0 * L * (L + 2.0) * std::min(8.0, nt);
    S.lists += weight * (nt * (sizeof(PairTile) + 4 * sizeof(PairSlot) + sizeof(PairGroup) / 4 + 4) +
                         8.0 * sizeof(PairSeg) + sizeof(PairTarget) + sizeof(SphereParts));
    for (auto &T : of_target) {
        const double m = std::max(T.Ls, T.Lt);
        S.flops += weight * 21.0 * m * m * m;
        S.NL = std::max(S.NL, std::max(T.Ls, T.Lt));
    }
    for (auto &q : quads) S.nodes.insert(q.first);
}

double PairSize::shared() const {
    double b = 8.0 * (double)pair_delta_off_host(NL + 1);
    for (int q : nodes) b += 8.0 * (double)quad_size(NL, q) + 16.0 * q;
    return b;
}

int pair_finalize(ifs_ctx *c, PairBatch &B, std::vector<Task> &tasks, const char *name) {
    static const char *p2p[4] = {"p2p_gen_tables", "p2p_rot_fwd", "p2p_axial", "p2p_rot_back"};
    if (std::string(name) == "p2p")
        for (int i = 0; i < 4; ++i) B.pn[i] = p2p[i];
    B.tasks.swap(tasks);
    for (auto &T : B.tasks) B.NL = std::max(B.NL, std::max(T.Ls, T.Lt));
    std::map<int, int64_t> quads;
    build_tiles(B, quads);
    // nodes and weights of every set first, then the matrices
    std::map<int, int64_t> at;
    std::vector<double> nodes, mu, w;
    for (auto &q : quads) {
        at[q.first] = (int64_t)nodes.size();
        gauss_legendre(q.first, mu, w);
        nodes.insert(nodes.end(), mu.begin(), mu.end());
        nodes.insert(nodes.end(), w.begin(), w.end());
    }
    int64_t nq = (int64_t)nodes.size();
    for (auto &q : quads) {
        q.second = nq;
        nq += (int64_t)quad_size(B.NL, q.first);
    }
    int64_t tab = 0, ax = 0;
    for (size_t t = 0; t < B.tiles.size(); ++t) {
        PairTile &T = B.tiles[t];
        if (T.Q) {
            T.off_q = quads[T.Q];
            T.off_mu = at[T.Q];
        }
        tab += 4LL * T.tabw;
        for (int s = 0; s < 4 && !T.Q; ++s)
            if (B.slots[4 * t + s].src >= 0) ax += ax_size(T.Lt, B.slots[4 * t + s].Ls, B.slots[4 * t + s].K);
    }
    int rc;
    const size_t nd = (size_t)pair_delta_off_host(B.NL + 1);
    if ((rc = B.d_quad.alloc(8 * (size_t)std::max<int64_t>(nq, 2))) || (rc = B.d_delta.alloc(8 * nd))) return rc;
    if (!nodes.empty() && hipMemcpy(B.d_quad.p, nodes.data(), 8 * nodes.size(), hipMemcpyHostToDevice) != hipSuccess)
        return IFS_E_HIP;
    launch_pair_delta(B.NL, B.d_delta.as<double>(), nd, c->stream);
    for (auto &q : quads)
        launch_pair_quad(B.NL, q.first, B.d_quad.as<double>() + at[q.first], B.d_quad.as<double>() + q.second,
                         quad_size(B.NL, q.first), c->stream);
    if (hipPeekAtLastError() != hipSuccess) return IFS_E_HIP;
    const size_t need = 16 * (size_t)(tab + ax);
    B.kept = need + c->ws_cached <= c->cache_budget;
    if (B.kept) {
        if ((rc = B.own_tab.alloc(16 * (size_t)tab)) || (rc = B.own_ax.alloc(16 * (size_t)std::max<int64_t>(ax, 1))))
            return rc;
        c->ws_cached += need;
    }
    return pair_plan(c, B);
}

bool pair_parts(const ifs_ctx *c, const PairBatch &B, int nrhs) {
    return B.d_parts.p && pair_group(c, B, nrhs) == nrhs;
}

int pair_prepare(ifs_ctx *c, const PairBatch &B, int nrhs) {
    return ws_reserve(c, pair_need(B, pair_group(c, B, nrhs)));
}

int pair_run(ifs_ctx *c, PairBatch &B, const double2 *src_pool, double2 *dst_pool, int nrhs, int64_t src_stride,
             int64_t dst_stride) {
    const int group = pair_group(c, B, nrhs);
    const bool parts = pair_parts(c, B, nrhs);
    if (int rc = pair_prepare(c, B, nrhs)) return rc;
    const PairTile *tiles = B.d_tiles.as<PairTile>();
    const PairSlot *slots = B.d_slots.as<PairSlot>();
    const PairSeg *segs = B.d_segs.as<PairSeg>();
    const double *quad = B.d_quad.as<double>(), *delta = B.d_delta.as<double>();
    double2 *tab = B.kept ? B.own_tab.as<double2>() : c->ws_d.as<double2>();
    double2 *wax = B.kept ? B.own_ax.as<double2>() : c->ws_ax.as<double2>();
    double *Y = c->ws_y.as<double>(), *Z = c->ws_z.as<double>();
    double2 *W = c->ws_s.as<double2>();
    for (auto &ch : B.chunks) {
        const int nt = ch.t1 - ch.t0;
        if (!(B.kept && B.ready)) {
            Scope s(c, B.pn[0]);
            launch_pair_tables(tiles, slots, ch.t0, nt, ch.max_P, quad, tab, c->stream);
            if (ch.c1 > ch.c0) {
                const Task *tk = B.d_close.as<Task>() + ch.c0;
                launch_gen_sect(tk, ch.c1 - ch.c0, ch.max_nmax, c->ws_s.as<double2>(), c->stream);
                launch_gen_axial(tk, ch.c1 - ch.c0, ch.maxK_close, ch.max_nmax, c->ws_s.as<double2>(), wax, c->stream);
            }
        }
        for (int r0 = 0; r0 < nrhs; r0 += group) {
            const int nr = std::min(group, nrhs - r0);
            {
                Scope s(c, B.pn[1], ch.f_fwd * nr);
                launch_pair_fwd(tiles, slots, ch.t0, nt, ch.max_Ls, delta, tab, src_pool + r0 * src_stride, src_stride,
                                Y, ch.n_y, nr, c->stream);
            }
            {
                Scope s(c, B.pn[2], ch.f_ax * nr);
                launch_pair_axial(tiles, slots, B.d_groups.as<PairGroup>() + ch.a0, ch.a1 - ch.a0,
                                  B.d_order.as<int32_t>(), ch.waves, ch.max_K, std::max(ch.max_Ls, ch.max_Lt), B.NL,
                                  quad, tab, wax, Y, ch.n_y, Z, ch.n_z, nr, c->stream);
            }
            {
                Scope s(c, B.pn[3], ch.f_back * nr);
                launch_pair_back(tiles, segs, ch.s0, ch.s1 - ch.s0, ch.max_Lt, delta, tab, Z, ch.n_z, W, ch.n_w, nr,
                                 c->stream);
                if (!parts)
                    launch_pair_reduce(B.d_targets.as<PairTarget>(), segs, ch.g0, ch.g1 - ch.g0, ch.max_Lt, W, ch.n_w,
                                       dst_pool + r0 * dst_stride, dst_stride, nr, c->stream);
            }
        }
    }
    if (hipPeekAtLastError() != hipSuccess) return IFS_E_HIP;
    if (B.kept && !B.ready) B.ready = !capturing(c);
    return IFS_OK;
}

uint64_t pair_sig(const PairBatch &B) {
    uint64_t h = 0;
    for (const DevBuf *d : {&B.d_tiles, &B.d_slots, &B.d_segs, &B.d_targets, &B.d_parts, &B.d_close, &B.d_groups,
                            &B.d_order, &B.d_delta, &B.d_quad, &B.own_tab, &B.own_ax})
        h ^= (uint64_t)(uintptr_t)d->p + 0x9e3779b97f4a7c15ull + (h << 6) + (h >> 2);
    return h;
}

}  // namespace ifs
