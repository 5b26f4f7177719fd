// Level-synchronous driver of the MI355X INSCY engine (every mode; the trees'
// paths or, in a permuted level order, chains: inscy_perm.hip).
//
// In the reference's depth-first recursion (INSCYCPU3Weak,
// src/algorithms/inscy/InscyNodeCpu.cu:159-235) only pruneRedundancy and join
// read the result built so far.  restrict, mergeWithNeighbors, the
// weak-density prune and the s-connection prune read nothing but the parent
// tree, and the dense components of a subspace read nothing but the data.  So
// the tree of restricted trees is grown here one level at a time:
//   - all trees of a level get their merge flags in one pass and one read-back;
//   - the level's child subspaces go through in batches: one grid-index build,
//     one neighbour-count pass over the trees' points, one partition pass of
//     every (tree, dimension) pair and one read-back of the group sizes;
//   - the surviving children of a batch get their path prune, and their new
//     subspaces their dense components, a handful of launches for all of them.
// pruneRedundancy and join are then replayed on the device in stages that keep
// the reference's depth-first order wherever it matters (steps on subspaces
// one of which contains the other), which gives the depth-first recursion's
// result exactly.

#include "inscy_engine.h"

#include <functional>

namespace inscy {

namespace {
// child subspaces per batch (inscy_set_tuning, INSCY_MAX_BATCH override; the
// memory budget bounds them first unless n is small): every batch costs about 20
// launches, a wait and a read-back (n=20,011 d=70, 49,000 child subspaces:
// batches of 1024 118.3 ms, 2048 112.2, 4096 107.6, 8192 107.3)
constexpr size_t kMaxBatch = 4096;
inline int nblocks(long long count) { return (int) ((count + kBlockThreads - 1) / kBlockThreads); }
}  // namespace

void Engine::put(void *dst, const void *src, size_t bytes) {
    if (!bytes) return;
    const size_t need = (bytes + 255) & ~(size_t) 255;
    if (up_top + need > up.cap) {
        const bool defer = up_defer;
        if (up_top > 0) sync();  // staged copies still read the buffer (sync issues a deferred one)
        up_defer = defer;
        up_top = 0;
        if (need > up.cap) up.get(std::max(need, 2 * up.cap));
    }
    std::memcpy(up.p + up_top, src, bytes);
    if (up_defer) {
        // pool takes and staging places are both rounded to 256 bytes, so a
        // contiguous pair extends the pending copy (over the padding between
        // them, which lies inside the earlier take)
        const size_t padded = (pend_bytes + 255) & ~(size_t) 255;
        if (pend_bytes && static_cast<char *>(dst) == pend_dst + padded && up_top == pend_src + padded) {
            pend_bytes = padded + bytes;
        } else {
            if (pend_bytes) HIP_OK(hipMemcpyAsync(pend_dst, up.p + pend_src, pend_bytes, hipMemcpyHostToDevice, st));
            pend_dst = static_cast<char *>(dst);
            pend_src = up_top;
            pend_bytes = bytes;
        }
    } else {
        HIP_OK(hipMemcpyAsync(dst, up.p + up_top, bytes, hipMemcpyHostToDevice, st));
    }
    up_top += need;
}

void Engine::run_levels(inscy_result &out) {
    lt.clear();
    emask.clear();
    col_base = 0;
    col_feat.clear();
    col_tree.clear();
    col_m.clear();
    col_child0.clear();
    col_G.clear();
    store.chunk = (size_t) 256 << 20;
    batch.chunk = (size_t) 256 << 20;
    up.get((size_t) 4 << 20);
    max_batch = kMaxBatch;
    if (const char *e = std::getenv("INSCY_MAX_BATCH")) max_batch = (size_t) std::max(1, std::atoi(e));
    if (max_batch_override > 0) max_batch = (size_t) max_batch_override;
    batch_budget = (size_t) 2 << 30;
    if (available) batch_budget = std::min<size_t>(std::max<size_t>(available / 8, (size_t) 256 << 20), (size_t) 8 << 30);
    kept.clear();
    keptp.reset();
    kept_used = 0;
    kept_budget = keep_budget_override >= 0 ? (size_t) keep_budget_override : batch_budget;
    if (batch_budget_override > 0) batch_budget = (size_t) batch_budget_override;
    colp.reset();
    cols_used = 0;

    // the root tree: every point, the root s-connection paths
    Pool &L0 = lvl[cur_lvl];
    lvl[cur_lvl ^ 1].reset();
    int *P = store.take<int>(n);
    int *cnt0 = reinterpret_cast<int *>(small + 1);  // zeroed by the set-up
    LTree root;
    root.first = 0;
    root.pass = true;
    root.W = P;
    root.nW = n;
    root.pre = n;
    // identity order: a path per point; permuted: a chain per near-edge dimension
    // (positions in the lists are ints: tables that could hold more chains are counted first)
    size_t most = permuted ? (size_t) n * d : (size_t) n;
    if (most > (size_t) chain_limit) {
        unsigned long long *total = small + 2;  // zeroed by the set-up
        HIP_OK(launch_p_chains(nearm, n, total, st));
        unsigned long long *h = reinterpret_cast<unsigned long long *>(down.get(sizeof(*h)));
        HIP_OK(hipMemcpyAsync(h, total, sizeof(*h), hipMemcpyDeviceToHost, st));
        sync();
        if (*h > (unsigned long long) chain_limit)
            throw Failure(INSCY_ERR_UNSUPPORTED, "more than 2^31 - 1 s-connection chains in a permuted level order");
        most = (size_t) *h;
    }
    root.spx = L0.take<int>(most);
    root.spm = L0.take<uint64_t>(most * pw);
    root.nsp_max = (int) most;
    root.slot = 0;
    HIP_OK(dev_alloc(&edges, ((size_t) ecells + 3) * sizeof(float)));
    if (permuted)
        HIP_OK(launch_p_root(nearm, n, d, P, root.spx, root.spm, cnt0, ecells, edges, st));
    else
        HIP_OK(launch_b_root(nearm, n, P, root.spx, root.spm, mw, cnt0, ecells, edges, st));
    lt.push_back(std::move(root));
    stats.calls = 1;

    auto t0 = std::chrono::steady_clock::now();
    std::vector<int> frontier{0};
    const int *counts = cnt0;
    while (!frontier.empty()) {
        expand_level(frontier, counts);
        frontier.swap(lv_next);
        counts = lv_next_counts;
        lvl[cur_lvl].reset();
        cur_lvl ^= 1;
    }

    // children in the reference's visiting order: dimension, then cell group
    for (auto &t : lt)
        std::stable_sort(t.kids.begin(), t.kids.end(), [&](int a, int b) {
            return lt[a].m != lt[b].m ? lt[a].m < lt[b].m : lt[a].lo < lt[b].lo;
        });
    sync();
    batch_most = batch.most;
    auto t1 = std::chrono::steady_clock::now();
    // superset rows of every subspace with a row: AND of per-dimension bitsets
    {
        const int ne = (int) emask.size();
        const int words = (ne + 63) / 64;
        std::vector<std::vector<uint64_t>> has(d, std::vector<uint64_t>(words, 0));
        for (int e = 0; e < ne; ++e)
            for (int k = 0; k < d; ++k)
                if (dhas(emask[e], k)) has[k][e >> 6] |= 1ull << (e & 63);
        std::vector<int> flat;
        std::vector<uint64_t> acc(words);
        sup_at.clear();
        for (int e = 0; e < ne; ++e) {
            const dmask_t sm = emask[e];
            std::fill(acc.begin(), acc.end(), ~0ull);
            for (int k = 0; k < d; ++k)
                if (dhas(sm, k))
                    for (int w = 0; w < words; ++w) acc[w] &= has[k][w];
            const int at = (int) flat.size();
            for (int w = 0; w < words; ++w)
                for (uint64_t b = acc[w]; b; b &= b - 1) flat.push_back(w * 64 + __builtin_ctzll(b));
            sup_at[sm] = {at, (int) flat.size() - at};
        }
        d_sup = upload(store, flat);
        sup_flat.swap(flat);
    }
    keepv = store.take<int>(lt.size());
    rep_join = 0;
    replay_staged();
    if (collect) finish_collect(out);
    sync();
    auto t2 = std::chrono::steady_clock::now();
    if (trace_on) {
        std::vector<int> keep(lt.size());
        HIP_OK(hipMemcpyAsync(keep.data(), keepv, keep.size() * sizeof(int), hipMemcpyDeviceToHost, st));
        sync();
        trace.clear();
        trace_tree(0, keep);
    }
    auto t3 = std::chrono::steady_clock::now();
    if (batch_trace)
        std::fprintf(stderr, "[inscy pairs] %lld (tree, dimension) pairs, %lld with a surviving child; "
                             "points counted %lld, in pairs with a surviving child %lld; pairs whose largest "
                             "cell group holds fewer than min_size points %lld (points %lld)\n",
                     pair_stats[0], pair_stats[1], pair_stats[2], pair_stats[3], pair_stats[4], pair_stats[5]);
    emit(out);
    stats.expand_seconds = std::chrono::duration<double>(t1 - t0).count();
    stats.replay_seconds = std::chrono::duration<double>(t2 - t1).count();
    stats.emit_seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t3).count();
}

// One level: merge flags and exact path counts of the frontier, then the
// child subspaces in batches.  Fills lv_next (surviving children that can
// still restrict) and lv_next_counts (their path counters).
void Engine::expand_level(const std::vector<int> &frontier, const int *counts) {
    Pool &cur = lvl[cur_lvl];
    Pool &nxt = lvl[cur_lvl ^ 1];
    lv_next.clear();
    lv_nslots = 0;
    lv_next_counts = nullptr;
    lv_act.clear();
    for (int t : frontier)
        if (lt[t].first < d) lv_act.push_back(t);
    if (lv_act.empty()) return;
    const int na = (int) lv_act.size();

    // merge flags of every dimension >= first of every tree
    std::vector<FlagTree> ft(na);
    std::vector<int> fblk(na + 1, 0);
    lv_gidoff.assign(na, 0);
    int ftot = 0;
    for (int a = 0; a < na; ++a) {
        const LTree &t = lt[lv_act[a]];
        ft[a] = FlagTree{t.spx, t.spm, counts + t.slot, t.first, ftot, mw};
        lv_gidoff[a] = ftot;
        ftot += (d - t.first) * cells;
        fblk[a + 1] = fblk[a] + nblocks(t.nsp_max);
    }
    int *flags = cur.take<int>(ftot);
    lv_next_counts = nxt.take<int>(ftot);  // at most one child per cell
    FillMany fill;
    fill.add(flags, 0, (size_t) ftot * sizeof(int));
    fill.add(lv_next_counts, 0, (size_t) ftot * sizeof(int));
    HIP_OK(launch_fill_many(fill, st));
    defer_uploads();
    FlagTree *dft = upload(cur, ft);
    int *dfb = upload(cur, fblk);
    flush_uploads();
    HIP_OK((permuted ? launch_p_flags : launch_b_flags)(dft, dfb, na, fblk[na], cellC, n, cells, flags, st));
    const int nf = (int) frontier.size();
    char *h = down.get((size_t) (ftot + nf) * sizeof(int));
    HIP_OK(hipMemcpyAsync(h, flags, (size_t) ftot * sizeof(int), hipMemcpyDeviceToHost, st));
    HIP_OK(hipMemcpyAsync(h + (size_t) ftot * sizeof(int), counts, (size_t) nf * sizeof(int), hipMemcpyDeviceToHost,
                          st));
    sync();
    const int *hf = reinterpret_cast<const int *>(h);
    const int *hc = hf + ftot;
    int max_slot = -1;
    for (int t : frontier) max_slot = std::max(max_slot, lt[t].slot);
    if (max_slot >= nf) throw Failure(INSCY_ERR_DEVICE, "internal: path counter slot out of range");
    for (int t : frontier) lt[t].nsp = std::min(hc[lt[t].slot], lt[t].nsp_max);

    // cell groups (restrict + mergeWithNeighbors, ScyTreeNode.cu:837-851)
    lv_groups.assign(na, {});
    std::vector<int> gid(ftot);
    for (int a = 0; a < na; ++a) {
        const LTree &t = lt[lv_act[a]];
        lv_groups[a].resize(d - t.first);
        for (int m = t.first; m < d; ++m) {
            const int *f = hf + lv_gidoff[a] + (m - t.first) * cells;
            int *gm = gid.data() + lv_gidoff[a] + (m - t.first) * cells;
            auto &gs = lv_groups[a][m - t.first];
            for (int c = 0; c < cells; ++c) {
                int lo = c;
                while (f[c] && c < cells - 1) ++c;
                for (int x = lo; x <= c; ++x) gm[x] = (int) gs.size();
                gs.push_back({lo, c});
            }
        }
    }
    lv_gid = upload(cur, gid);
    lv_skip.clear();
    if (pruner || collect) score_pairs(na);

    // child subspaces: per run of frontier trees with one mask, S | {m} for m >= first
    std::vector<ChildSub> cs;
    std::set<dmask_t> seen;
    for (int a = 0; a < na;) {
        int b = a;
        while (b < na && lt[lv_act[b]].smask == lt[lv_act[a]].smask) ++b;
        const LTree &t = lt[lv_act[a]];
        // the trees of one mask are created together, so each child subspace
        // is reached from exactly one run
        if (!seen.insert(t.smask).second) throw Failure(INSCY_ERR_DEVICE, "internal: frontier masks not grouped");
        for (int m = t.first; m < d; ++m) {
            bool any = false;  // some pair of this child subspace is not skipped
            for (int x = a; x < b && !any; ++x) any = pair_on(x, m);
            if (any) cs.push_back({t.smask | dbit(m), m, a, b});
        }
        a = b;
    }

    // batches bounded by memory, count and 32-bit positions
    const bool fan = fan_level(cs);
    size_t i = 0;
    while (i < cs.size()) {
        size_t j = i;
        size_t bytes = 0;
        long long hsum = 1;
        while (j < cs.size() && j - i < max_batch) {
            const ChildSub &c = cs[j];
            SubspaceArg S = arg_of(c.s);
            GridArg G = grid_of(S, -1, true);
            const long long ncell = grid_cells(G);
            // process_batch's takes per subspace: counts, query flags and
            // list, two sample edges, sample-phase roots and parents (25 bytes a
            // point), an index that is not kept (keys, rank, order, position:
            // 16, k coordinate columns: 4k, grid histogram and offsets), the
            // phi pass's queue (8)
            size_t est = (size_t) n * (41 + 4 * (size_t) S.k + (phi_mode ? 8 : 0)) + (size_t) ncell * 12;
            // the index and the queries (learned: and their trees) of a fanned mask
            if (fan && (j == i || cs[j - 1].t0 != c.t0))
                est += (size_t) n * (21 + (pruner ? 4 : 0) + 4 * (size_t) S.k) + (size_t) ncell * 12;
            for (int a = c.t0; a < c.t1; ++a) {
                if (!pair_on(a, c.m)) continue;
                const LTree &t = lt[lv_act[a]];
                // lists, and the path prune's table (a few branch levels per path)
                est += (size_t) t.nW * 8 + (size_t) t.nsp * (12 + 32 * std::min<size_t>(d - 1 - c.m, 4)) + 8 * 256 * 4;
                // the point filter's table and flags, the routed chains and their table
                if (permuted) est += (size_t) t.nW * 33 + (size_t) t.nsp * 96;
            }
            const bool fits = bytes + est <= batch_budget && (long long) (j - i + 1) * n < INT_MAX &&
                              hsum + ncell < INT_MAX;
            if (j > i && !fits) break;
            bytes += est;
            hsum += ncell;
            ++j;
        }
        process_batch(cs, i, j, fan);
        i = j;
    }
}

// Grid index of the child subspace S | {m} (m its last dimension): S's own
// index where it costs the neighbour passes little (S's index dimensions are at
// most 25% less selective than the best ones of S | {m}; expected candidates
// per query scale with the product of the index dimensions' selectivity
// scores), so that the children of one frontier mask read one sort and one set
// of columns.
GridArg Engine::child_grid(const SubspaceArg &S) const {
    const GridArg gopt = grid_of(S, -1, true);
    const int kS = S.k - 1;
    if (kS < 3 || __builtin_popcountll(match_of(S) & ((1ull << kS) - 1)) < 3) return gopt;
    const GridArg gbest = grid_of(S, S.k - 1, true);
    double cs = 1.0, co = 1.0;
    for (int a = 0; a < gbest.j; ++a) cs *= std::max(score[S.dims[gbest.tI[a]]], 1.0);
    for (int a = 0; a < gopt.j; ++a) co *= std::max(score[S.dims[gopt.tI[a]]], 1.0);
    return gbest.j == gopt.j && cs <= 1.25 * co ? gbest : gopt;
}

// The grid indexes (order, pos, off) and coordinate columns of the subspaces
// hs, whose S and G are set: a sort or column the run has kept is used where it
// lies, the others are sorted and gathered here, into kept memory while the
// budgets last, else into the batch's.  ctab receives the column pointers
// (S.k per subspace, in order); the caller uploads it and sets hs[b].col.
void Engine::index_of(std::vector<BatchSub> &hs, std::vector<const float *> &ctab) {
    std::vector<SortJob> sorts;
    std::vector<ColJob> cols;
    long long hmiss = 0;
    int max_cell = 0;
    for (BatchSub &x : hs) {
        uint64_t key = (uint64_t) x.G.j;
        for (int a = 0; a < x.G.j; ++a) key |= (uint64_t) (x.S.dims[x.G.tI[a]] + 1) << (8 * (a + 1));
        Sort *srt = nullptr;
        auto it = kept.find(key);
        if (it != kept.end()) {
            srt = &it->second;
            stats.sorts_kept++;
        } else if (auto jt = batch_sorts.find(key); jt != batch_sorts.end()) {
            srt = &jt->second;
        } else {
            const int ncell = (int) grid_cells(x.G);
            const size_t need = ((size_t) 2 * n + ncell + 5) * sizeof(int) + 768;
            const bool keep = kept_used + need <= kept_budget;
            Pool &pool = keep ? keptp : batch;
            Sort s;
            s.keep = keep;
            s.order = pool.take<int>((size_t) n + 4);  // the grouped walks read up to 3 ids past a run
            s.pos = pool.take<int>(n);
            s.off = pool.take<int>((size_t) ncell + 1);
            if (keep) {
                kept_used += need;
                s.col.assign(d, nullptr);
            }
            SortJob j{};
            j.order = s.order;
            j.pos = s.pos;
            j.off = s.off;
            j.hoff = hmiss;
            j.j = x.G.j;
            j.C = x.G.C;
            j.F = x.G.F;
            j.ncell = ncell;
            for (int a = 0; a < x.G.j; ++a) j.dims[a] = x.S.dims[x.G.tI[a]];
            hmiss += ncell;
            max_cell = std::max(max_cell, ncell);
            sorts.push_back(j);
            srt = &(keep ? kept : batch_sorts).emplace(key, std::move(s)).first->second;
        }
        x.order = srt->order;
        x.pos = srt->pos;
        x.off = srt->off;
        for (int t = 0; t < x.S.k; ++t) {
            const int dim = x.S.dims[t];
            float *c = srt->keep ? srt->col[dim] : nullptr;
            if (!c) {
                const size_t need = ((size_t) n + 4) * sizeof(float) + 256;
                const uint64_t ck = key | (uint64_t) (dim + 1) << 32;
                if (srt->keep && cols_used + need <= kept_budget) {
                    c = srt->col[dim] = colp.take<float>((size_t) n + 4);  // walks read up to 3 past the end
                    cols_used += need;
                    cols.push_back({srt->order, Xt + (size_t) dim * n, c});
                } else {
                    float *&bc = batch_cols[ck];
                    if (!bc) {
                        bc = batch.take<float>((size_t) n + 4);
                        cols.push_back({srt->order, Xt + (size_t) dim * n, bc});
                    }
                    c = bc;
                }
            }
            ctab.push_back(c);
        }
    }
    if (sorts.empty() && cols.empty()) return;
    const int ns = (int) sorts.size(), nc = (int) cols.size();
    defer_uploads();
    SortJob *ds = ns ? upload(batch, sorts) : nullptr;
    ColJob *dc = nc ? upload(batch, cols) : nullptr;
    flush_uploads();
    if (ns) {
        int *keys = batch.take<int>((size_t) ns * n), *rank = batch.take<int>((size_t) ns * n);
        int *hist = batch.take<int>(hmiss + 1), *off = batch.take<int>(hmiss + 1);
        const size_t sb = scan_temp_bytes((int) (hmiss + 1));
        char *tmp = batch.take<char>(sb);
        HIP_OK(launch_b_sort(D, ds, ns, (int) hmiss, max_cell, keys, rank, hist, off, tmp, sb, st));
    }
    if (nc) HIP_OK(launch_b_gather(dc, nc, n, st));
}

// Whether the level's children are counted by one walk per frontier mask
// (k_b_fan) instead of one per child: when the mask's own grid index has as
// many dimensions as its children's, so that the walk meets no more candidates
// than each child's would.  Where the children's index has one more (masks of
// two dimensions whose cells cubed still fit the grid), a walk per child meets
// far fewer: n=100,000 d=20, masks of two dimensions 16.8 ms by child, 39 ms by
// mask; n=25,000 d=15, eps=0.015 (two index dimensions at most) 2.19 and 1.74.
bool Engine::fan_level(const std::vector<ChildSub> &cs) const {
    if (cs.empty() || n >= kFanPoints || (long long) n * d >= 1ll << 30) return false;  // 32-bit offsets into X
    if (permuted) return false;  // the children match different dimensions of one mask
    if (walk_per_child) return false;
    const SubspaceArg S = arg_of(cs[0].s & ~dbit(cs[0].m));
    if (S.k < 1 || S.k > kMaxFastK) return false;
    return grid_of(S, -1, true).j >= grid_of(arg_of(cs[0].s), -1, true).j;
}

void Engine::process_batch(const std::vector<ChildSub> &cs, size_t i0, size_t i1, bool fan) {
    Pool &nxt = lvl[cur_lvl ^ 1];
    batch.reset();
    batch_sorts.clear();
    batch_cols.clear();
    const int B = (int) (i1 - i0);
    const int k = dcount(cs[i0].s);  // of every child: the level's trees restrict equally many dimensions
    const int kfast = !generic_walk && k <= kMaxFastK ? k : 0;

    // ---- the batch's child subspaces
    std::vector<BatchSub> hs(B);
    int *cntB = batch.take<int>((size_t) B * n);
    for (int b = 0; b < B; ++b) {
        const ChildSub &c = cs[i0 + b];
        BatchSub &x = hs[b];
        std::memset(&x, 0, sizeof(x));
        x.S = arg_of(c.s);
        x.base = x.nbase = (long long) b * n;
        x.cnt = cntB + (size_t) b * n;
        x.cap = cap_of(k);
        x.thr_dense = dense_thr[k];
        set_bounds(c.s, x);
        x.dbit = phi_mode ? 2 : 0;
        x.matchmask = match_of(x.S);
        x.phi_w = phi_weak;
        x.phi_d = phi_dense[k];
        if (!fan) x.G = child_grid(x.S);
    }

    // ---- the walked subspaces: every child, or with `fan` every frontier
    // mask, whose walk serves all its children; their queries are the points
    // of the trees refined, in sorted order
    std::vector<BatchSub> gs;       // fan: the masks
    constexpr int kWidths[] = {4, 8, 16, 32, kFanMost};
    std::vector<FanJob> jobs[5];    // by the width of their walk
    std::vector<QuerySeg> qs;
    std::vector<int> qblk{0};
    std::vector<unsigned long long> live;  // fan: FanTable::live of the segments
    bool skips = false;                    // fan: some segment has a pair that is not
    long long qoff = 0;
    auto add_segment = [&](int w, int a) {
        const LTree &t = lt[lv_act[a]];
        if (t.nW <= 0) return false;
        qs.push_back({t.W, t.nW, w});
        qblk.push_back(qblk.back() + nblocks(t.nW));
        qoff += t.nW;
        return true;
    };
    if (fan) {
        for (int b = 0; b < B;) {
            const ChildSub &c = cs[i0 + b];
            int e = b;
            while (e < B && cs[i0 + e].t0 == c.t0) ++e;
            BatchSub g;
            std::memset(&g, 0, sizeof(g));
            g.S = arg_of(c.s & ~dbit(c.m));
            g.G = grid_of(g.S, -1, true);
            g.base = (long long) gs.size() * n;
            long long qmax = 0;
            for (int a = c.t0; a < c.t1; ++a) {
                if (!lv_skip.empty()) {
                    // the tree's live pairs among the mask's children
                    unsigned long long on[2] = {0, 0};
                    int dead = 0;
                    for (int x = b; x < e; ++x) {
                        if (pair_on(a, cs[i0 + x].m))
                            on[(x - b) / kFanMost] |= 1ull << ((x - b) % kFanMost);
                        else
                            ++dead;
                    }
                    if (dead == e - b || lt[lv_act[a]].nW <= 0) continue;
                    live.insert(live.end(), on, on + 2);
                    skips |= dead > 0;
                }
                if (add_segment((int) gs.size(), a)) qmax += lt[lv_act[a]].nW;
            }
            g.qmax = (int) qmax;
            for (int at = b; at < e; at += kFanMost) {
                const int nch = std::min(kFanMost, e - at);
                int w = 0;
                while (kWidths[w] < nch) ++w;
                jobs[w].push_back({(int) gs.size(), at, nch, (at - b) / kFanMost});
            }
            gs.push_back(g);
            b = e;
        }
    } else {
        for (int b = 0; b < B; ++b) {
            const ChildSub &c = cs[i0 + b];
            long long qmax = 0;
            for (int a = c.t0; a < c.t1; ++a)
                if (pair_on(a, c.m) && add_segment(b, a)) qmax += lt[lv_act[a]].nW;
            hs[b].qmax = (int) qmax;
        }
    }
    std::vector<BatchSub> &ws = fan ? gs : hs;
    const int nw = (int) ws.size();
    std::vector<const float *> ctab;
    index_of(ws, ctab);

    BatchIndex X{};
    X.edge = edges;
    X.qflag = batch.take<uint8_t>(((size_t) nw * n + 15) & ~(size_t) 15);  // read 16 bytes a lane
    X.qlist = batch.take<int>(std::max<long long>(qoff, 1));
    X.nsel = batch.take<int>(1);
    X.qstart = batch.take<int>(nw + 1);
    X.select_bytes = select_temp_bytes(nw * n);
    X.select_temp = batch.take<char>(X.select_bytes);
    X.nb = batch.take<int>((size_t) kSampleEdges * B * n);
    X.nfb = batch.take<int>(1);
    X.fbcap = phi_mode ? B * n : 1;  // each point of each subspace is sent at most once per pass
    X.fb = batch.take<int2>(X.fbcap);
    // ---- (tree, dimension) pairs to partition by the cell groups
    struct PairInfo {
        int a, b, G, cnt_off;
    };
    std::vector<PairInfo> pinfo;
    int pc_total = 0;
    for (int b = 0; b < B; ++b) {
        const ChildSub &c = cs[i0 + b];
        for (int a = c.t0; a < c.t1; ++a) {
            if (!pair_on(a, c.m)) continue;
            const LTree &t = lt[lv_act[a]];
            const int G = (int) lv_groups[a][c.m - t.first].size();
            pinfo.push_back({a, b, G, pc_total});
            pc_total += 8 * G;
        }
    }
    int *pcnt = batch.take<int>(std::max(pc_total, 1));
    FillMany fill;
    // permuted order: the restriction of every pair, and the point filters
    std::vector<PermStep> steps;
    std::vector<PermFilter> filters;
    std::vector<int> filter_of(permuted ? pinfo.size() : 0, -1), fltblk{0};
    if (permuted) {
        size_t slots_total = 0;
        std::vector<size_t> slots_at;
        for (size_t j = 0; j < pinfo.size(); ++j) {
            const ChildSub &c = cs[i0 + pinfo[j].b];
            const LTree &t = lt[lv_act[pinfo[j].a]];
            steps.push_back(perm_step(t.smask, c.m));
            // groups of one cell each keep every point
            if (!steps.back().filt || pinfo[j].G == cells || t.nW <= 0) continue;
            PermFilter f;
            std::memset(&f, 0, sizeof(f));
            f.s = steps.back();
            f.P = t.W;
            f.nP = t.nW;
            f.gid = lv_gid + lv_gidoff[pinfo[j].a] + (c.m - t.first) * cells;
            f.keep = batch.take<uint8_t>(t.nW);
            const size_t slots = path_slots(t.nW);
            f.tmask = (uint64_t) (slots - 1);
            slots_at.push_back(slots_total);
            slots_total += slots;
            filter_of[j] = (int) filters.size();
            filters.push_back(f);
            fltblk.push_back(fltblk.back() + nblocks(t.nW));
        }
        uint64_t *tables = batch.take<uint64_t>(slots_total);
        fill.add(tables, ~0u, slots_total * sizeof(uint64_t));
        for (size_t f = 0; f < filters.size(); ++f) filters[f].table = tables + slots_at[f];
    }
    fill.add(X.nb, ~0u, (size_t) kSampleEdges * B * n * sizeof(int));
    fill.add(cntB, ~0u, (size_t) B * n * sizeof(int));
    fill.add(X.qflag, 0, (size_t) nw * n);
    fill.add(pcnt, 0, (size_t) pc_total * sizeof(int));
    if (phi_mode && fan) fill.add(X.nfb, 0, sizeof(int));
    HIP_OK(launch_fill_many(fill, st));

    auto columns = [&](std::vector<BatchSub> &v, const std::vector<const float *> &tab) {
        const float *const *dcol = upload(batch, tab);
        size_t at = 0;
        for (BatchSub &x : v) {
            x.col = dcol + at;
            at += x.S.k;
        }
    };
    std::vector<int> cblk{0};
    FanTable ft{};
    defer_uploads();
    columns(ws, ctab);
    BatchSub *dws = upload(batch, ws);
    QuerySeg *dqs = upload(batch, qs);
    int *dqb = upload(batch, qblk);
    FanJob *djobs[5] = {};
    int *djb[5] = {}, njb[5] = {};
    BatchSub *dsubs = nullptr;  // fan: the children, for the phi recomputation
    int *dcb = nullptr;
    if (fan) {
        std::vector<int *> tc(B);
        std::vector<int> td(B);
        std::vector<long long> tbase(B);
        for (int b = 0; b < B; ++b) {
            tc[b] = hs[b].cnt;
            td[b] = cs[i0 + b].m;
            tbase[b] = hs[b].nbase;
        }
        ft = FanTable{upload(batch, tc), upload(batch, td), upload(batch, tbase), skips ? upload(batch, live) : nullptr,
                      skips ? batch.take<int>((size_t) nw * n) : nullptr};
        for (int w = 0; w < 5; ++w) {
            if (jobs[w].empty()) continue;
            std::vector<int> blk{0};
            for (const FanJob &j : jobs[w]) blk.push_back(blk.back() + (gs[j.g].qmax + kFanQueries - 1) / kFanQueries);
            djobs[w] = upload(batch, jobs[w]);
            djb[w] = upload(batch, blk);
            njb[w] = blk.back();
        }
        if (phi_mode) dsubs = upload(batch, hs);
    } else {
        for (int b = 0; b < B; ++b) cblk.push_back(cblk.back() + (hs[b].qmax + kQueriesPerBlock - 1) / kQueriesPerBlock);
        dcb = upload(batch, cblk);
    }
    flush_uploads();
    HIP_OK(launch_b_queries(dws, nw, n, dqs, dqb, (int) qs.size(), qblk.back(), X, const_cast<int *>(ft.seg), st));
    const bool dbg = batch_trace;
    std::chrono::steady_clock::time_point tq0, tq1;
    if (dbg) {
        sync();
        tq0 = std::chrono::steady_clock::now();
    }
    if (fan) {
        const KernelTimer tm = timer();
        if (tm.start) HIP_OK(hipEventRecord(tm.start, st));
        for (int w = 0; w < 5; ++w)
            HIP_OK(launch_b_fan(dws, djobs[w], djb[w], (int) jobs[w].size(), njb[w], kWidths[w], k - 1, ft, X, s_star,
                                prm.neighborhood_size, phi_mode, phi_all_exact, cap_of(k), phi_weak, phi_dense[k], D,
                                small + kStatAt, st));
        if (tm.stop) HIP_OK(hipEventRecord(tm.stop, st));
        if (phi_mode)
            HIP_OK(launch_phi_exact(D, dsubs, X.fb, X.nfb, X.fbcap, rank_perm, prm.neighborhood_size, s_star, st));
    } else {
        HIP_OK(launch_b_count(dws, B, dcb, cblk.back(), n, k, kfast, X, s_star, prm.neighborhood_size, phi_mode,
                              phi_all_exact, D, rank_perm, small + kStatAt, timer(), st));
    }
    if (dbg) {
        sync();
        tq1 = std::chrono::steady_clock::now();
    }

    // ---- partition of every (tree, dimension) pair by the cell groups
    const int np = (int) pinfo.size();
    std::vector<PartPair> pairs(np);
    std::vector<int> pblk(np + 1, 0);
    for (int j = 0; j < np; ++j) {
        const PairInfo &pi = pinfo[j];
        const ChildSub &c = cs[i0 + pi.b];
        const LTree &t = lt[lv_act[pi.a]];
        PartPair &pp = pairs[j];
        std::memset(&pp, 0, sizeof(pp));
        pp.P = t.W;
        pp.nP = t.nW;
        if (!permuted) {
            pp.spx = t.spx;
            pp.spm = t.spm;
            pp.nsp = t.nsp;
        } else if (filter_of[j] >= 0) {
            pp.keep = filters[filter_of[j]].keep;
        }
        pp.gid = lv_gid + lv_gidoff[pi.a] + (c.m - t.first) * cells;
        pp.weakcnt = hs[pi.b].cnt;
        pp.cnt = pcnt + pi.cnt_off;
        pp.outW = batch.take<int>(std::max(t.nW, 1));
        if (!permuted) {
            pp.outx = batch.take<int>(std::max(t.nsp, 1));
            pp.outm = batch.take<uint64_t>((size_t) std::max(t.nsp, 1) * mw);
        }
        pp.mw = mw;
        pp.m = c.m;
        pp.G = pi.G;
        pp.bp = nblocks((t.nW + kPartPerThread - 1) / kPartPerThread);
        pblk[j + 1] = pblk[j] + pp.bp + nblocks((pp.nsp + kPartPerThread - 1) / kPartPerThread);
    }
    std::vector<PermPair> ppairs(permuted ? np : 0);
    std::vector<int> ppblk(1, 0);
    for (int j = 0; j < (int) ppairs.size(); ++j) {
        const LTree &t = lt[lv_act[pinfo[j].a]];
        PermPair &pp = ppairs[j];
        pp = PermPair{steps[j], t.spx, t.spm, pairs[j].gid, pairs[j].cnt + 2 * pinfo[j].G, pairs[j].cnt + 6 * pinfo[j].G,
                      t.nsp, pinfo[j].G};
        ppblk.push_back(ppblk.back() + nblocks(t.nsp));
    }
    defer_uploads();
    PartPair *dpairs = upload(batch, pairs);
    int *dpb = upload(batch, pblk);
    PermFilter *dflt = permuted ? upload(batch, filters) : nullptr;
    int *dfltb = permuted ? upload(batch, fltblk) : nullptr;
    PermPair *dpp = permuted ? upload(batch, ppairs) : nullptr;
    int *dppb = permuted ? upload(batch, ppblk) : nullptr;
    flush_uploads();
    if (permuted) {
        HIP_OK(launch_p_filter(D, dflt, dfltb, (int) filters.size(), fltblk.back(), st));
        HIP_OK(launch_p_count(D, dpp, dppb, np, ppblk.back(), st));
    }
    HIP_OK(launch_b_partition(dpairs, dpb, np, pblk[np], cellC, n, weak_thr, phi_mode ? 1 : 0, prm.min_size, st));
    char *h = down.get((size_t) std::max(pc_total, 1) * sizeof(int));
    HIP_OK(hipMemcpyAsync(h, pcnt, (size_t) std::max(pc_total, 1) * sizeof(int), hipMemcpyDeviceToHost, st));
    sync();
    const std::vector<int> hcnt(reinterpret_cast<const int *>(h), reinterpret_cast<const int *>(h) + pc_total);

    // ---- children: trace rows, surviving trees, their point lists and path prunes
    std::vector<CopySeg> copies;
    std::vector<CopySeg> stamps;  // W points -> tree index, into the subspace's stamp array
    std::vector<int> stamp_b;
    std::vector<PruneChild> prune;
    std::vector<PermChild> pprune;
    std::vector<size_t> prune_slots;
    std::vector<char> passing(B, 0);
    size_t table_total = 0;
    for (int j = 0; j < np; ++j) {
        const PairInfo &pi = pinfo[j];
        const ChildSub &c = cs[i0 + pi.b];
        const int tparent = lv_act[pi.a];
        const int first = lt[tparent].first;
        const int G = pi.G;
        if (batch_trace) {
            bool any = false, big = false;
            for (int g = 0; g < G; ++g) {
                any |= hcnt[pi.cnt_off + G + g] >= prm.min_size;
                big |= hcnt[pi.cnt_off + g] >= prm.min_size;
            }
            pair_stats[0] += 1;
            pair_stats[1] += any;
            pair_stats[2] += lt[tparent].nW;
            pair_stats[3] += any ? lt[tparent].nW : 0;
            pair_stats[4] += big ? 0 : 1;
            pair_stats[5] += big ? 0 : lt[tparent].nW;
        }
        if (collect) {
            const long long gp = col_base + lv_pair0[pi.a] + (c.m - first);
            col_child0[gp] = (int) lt.size();
            col_G[gp] = G;
        }
        const int *c3 = hcnt.data() + pi.cnt_off;
        const unsigned long long *levels = reinterpret_cast<const unsigned long long *>(c3 + 6 * G);
        int offW = 0, offS = 0, others = 0;
        for (int g = 0; permuted && g < G; ++g) others += c3[6 * G + g];
        for (int g = 0; g < G; ++g) {
            const int nPr = c3[g], nW = c3[G + g];
            // permuted: the chains of the group's cells and of every other group's
            const int nSP = c3[2 * G + g] + (permuted ? others - c3[6 * G + g] : 0);
            LTree ch;
            ch.smask = c.s;
            ch.first = c.m + 1;
            ch.m = c.m;
            ch.lo = lv_groups[pi.a][c.m - first][g].lo;
            ch.hi = lv_groups[pi.a][c.m - first][g].hi;
            ch.pre = nPr;
            ch.nW = nW;
            ch.pass = nW >= prm.min_size;
            stats.trees++;
            if (ch.pass) {
                stats.calls++;
                passing[pi.b] = 1;
                int *Wst = store.take<int>(std::max(nW, 1));
                if (nW > 0) {
                    copies.push_back({pairs[j].outW + offW, Wst, nW, -1});
                    stamps.push_back({pairs[j].outW + offW, nullptr, nW, (int) lt.size()});
                    stamp_b.push_back(pi.b);
                }
                ch.W = Wst;
                if (ch.first < d) {
                    ch.slot = lv_nslots++;
                    ch.nsp_max = nSP;
                    ch.spx = nxt.take<int>(std::max(nSP, 1));
                    ch.spm = nxt.take<uint64_t>((size_t) std::max(nSP, 1) * pw);
                    if (nSP > 0 && permuted) {
                        const LTree &t = lt[tparent];
                        PermChild pc;
                        std::memset(&pc, 0, sizeof(pc));
                        pc.s = steps[j];
                        pc.spx = t.spx;
                        pc.chain = t.spm;
                        pc.gid = pairs[j].gid;
                        pc.P = t.W;
                        pc.keep = pairs[j].keep;
                        pc.weakcnt = pairs[j].weakcnt;
                        const size_t slots = path_slots(2 * (size_t) nSP);
                        pc.tmask = (uint64_t) (slots - 1);
                        pc.outx = ch.spx;
                        pc.outw = ch.spm;
                        pc.nout = lv_next_counts + ch.slot;
                        pc.nsp = t.nsp;
                        pc.nP = t.nW;
                        pc.nr = nSP;
                        pc.g = g;
                        pprune.push_back(pc);
                    } else if (nSP > 0) {
                        PruneChild pc;
                        std::memset(&pc, 0, sizeof(pc));
                        pc.smask = c.s;
                        const size_t slots = path_slots((size_t) levels[g]);
                        pc.tmask = (uint64_t) (slots - 1);
                        pc.W = pairs[j].outW + offW;
                        pc.spx = pairs[j].outx + offS;
                        pc.spm = pairs[j].outm + (size_t) offS * mw;
                        pc.mw = mw;
                        pc.outx = ch.spx;
                        pc.outm = ch.spm;
                        pc.nout = lv_next_counts + ch.slot;
                        pc.nW = nW;
                        pc.nsp = nSP;
                        prune_slots.push_back(table_total);
                        table_total += slots;
                        prune.push_back(pc);
                    }
                }
            }
            const int idx = (int) lt.size();
            const bool expand = ch.pass && ch.first < d;
            lt.push_back(std::move(ch));
            lt[tparent].kids.push_back(idx);
            if (expand) lv_next.push_back(idx);
            offW += nW;
            offS += nSP;
        }
    }

    // ---- permuted order: a chain passes to every surviving group, so what the
    // children's prunes take is known only here; as many children at a time as
    // fit a batch's bytes
    struct ChainPrune {
        std::vector<PermChild> c;
        std::vector<int> br{0}, bw{0}, bp{0};
        PermChild *dc;
        int *dbr, *dbw, *dbp;
    };
    auto chain_prune = [&](size_t c0, size_t c1, FillMany &f) {
        ChainPrune cp;
        cp.c.assign(pprune.begin() + c0, pprune.begin() + c1);
        size_t slots = 0, chains = 0;
        for (const PermChild &pc : cp.c) {
            slots += pc.tmask + 1;
            chains += pc.nr;
        }
        uint64_t *table = f.add(batch.take<uint64_t>(slots), ~0u, slots * sizeof(uint64_t));
        uint8_t *marks = f.add(batch.take<uint8_t>(2 * slots), 0, 2 * slots);
        dmask_t *bits = f.add(batch.take<dmask_t>(cp.c.size()), 0, cp.c.size() * sizeof(dmask_t));
        int *nr = f.add(batch.take<int>(cp.c.size()), 0, cp.c.size() * sizeof(int));
        int *rx = batch.take<int>(chains);
        uint64_t *rw = batch.take<uint64_t>(chains);
        for (PermChild &pc : cp.c) {
            pc.table = table;
            pc.marks = marks;
            pc.bits = bits++;
            pc.nr_at = nr++;
            pc.rx = rx;
            pc.rw = rw;
            table += pc.tmask + 1;
            marks += 2 * (pc.tmask + 1);
            rx += pc.nr;
            rw += pc.nr;
            cp.br.push_back(cp.br.back() + nblocks(pc.nsp));
            cp.bw.push_back(cp.bw.back() + nblocks((long long) pc.nP + pc.nr));
            cp.bp.push_back(cp.bp.back() + nblocks(pc.nr));
        }
        return cp;
    };
    auto upload_chains = [&](ChainPrune &cp) {
        cp.dc = upload(batch, cp.c);
        cp.dbr = upload(batch, cp.br);
        cp.dbw = upload(batch, cp.bw);
        cp.dbp = upload(batch, cp.bp);
    };
    auto prune_chains = [&](const ChainPrune &cp) {
        HIP_OK(launch_p_prune(D, cp.dc, (int) cp.c.size(), cp.dbr, cp.br.back(), cp.dbw, cp.bw.back(), cp.dbp,
                              cp.bp.back(), weak_thr, phi_mode ? 1 : 0, st));
    };
    size_t chains_from = 0;  // children whose prunes are left to the batch's last launches
    {
        size_t bytes = 0;
        for (size_t c = 0; c < pprune.size(); ++c) {
            const PermChild &pc = pprune[c];
            const size_t need = (size_t) pc.nr * 12 + (pc.tmask + 1) * 10 + sizeof(PermChild) + 32;
            if (c > chains_from && bytes + need > batch_budget) {
                const Pool::Mark mark = batch.mark();
                FillMany f;
                ChainPrune cp = chain_prune(chains_from, c, f);
                defer_uploads();
                upload_chains(cp);
                flush_uploads();
                HIP_OK(launch_fill_many(f, st));
                prune_chains(cp);
                batch.release(mark);  // stream order keeps the memory for the queued kernels
                chains_from = c;
                bytes = 0;
            }
            bytes += need;
        }
    }

    // ---- path prune of the surviving children, their point lists, and the
    // dense components of the subspaces that gained one: descriptors in one copy
    FillMany post;
    const int nprune = (int) prune.size();
    std::vector<int> bw(nprune + 1, 0), bp(nprune + 1, 0);
    ChainPrune chains;
    const bool any_chains = chains_from < pprune.size();
    if (any_chains) chains = chain_prune(chains_from, pprune.size(), post);
    if (nprune) {
        uint64_t *tables = post.add(batch.take<uint64_t>(table_total), ~0u, table_total * sizeof(uint64_t));
        dmask_t *bits = post.add(batch.take<dmask_t>(nprune), 0, (size_t) nprune * sizeof(dmask_t));
        for (int c = 0; c < nprune; ++c) {
            prune[c].table = tables + prune_slots[c];
            prune[c].bits = bits + c;
            bw[c + 1] = bw[c] + nblocks(prune[c].nW);
            bp[c + 1] = bp[c] + nblocks(prune[c].nsp);
        }
    }
    std::vector<BatchSub> hc;
    std::vector<Entry> ents;
    int ncomp = 0;
    for (int b = 0; b < B; ++b) ncomp += passing[b];
    std::vector<const float *> ctab2;
    if (ncomp > 0) {
        int *cntP = slabs.take<int>((size_t) ncomp * n);
        int *compP = slabs.take<int>((size_t) ncomp * n);
        int *csizeP = slabs.take<int>((size_t) ncomp * n);
        int *memP = slabs.take<int>((size_t) ncomp * n);
        uint8_t *inresP = post.add(slabs.take<uint8_t>((size_t) ncomp * n), 0, (size_t) ncomp * n);
        int *stampP = post.add(slabs.take<int>((size_t) ncomp * n), ~0u, (size_t) ncomp * n * sizeof(int));
        std::vector<int *> stamp_of(B, nullptr);
        grow_entries(nentries + ncomp);
        int ci = 0;
        for (int b = 0; b < B; ++b) {
            if (!passing[b]) continue;
            const dmask_t s = cs[i0 + b].s;
            BatchSub x = hs[b];
            x.base = (long long) ci * n;
            if (fan) x.G = child_grid(x.S);
            x.cnt = cntP + (size_t) ci * n;
            x.comp = compP + (size_t) ci * n;
            x.csize = csizeP + (size_t) ci * n;
            copies.push_back({hs[b].cnt, x.cnt, n, -1});
            hc.push_back(x);
            Subspace &sb = subs[s];
            sb.cnt = x.cnt;
            sb.comp = x.comp;
            sb.csize = x.csize;
            sb.inres = inresP + (size_t) ci * n;
            sb.tstamp = stampP + (size_t) ci * n;
            stamp_of[b] = sb.tstamp;
            sb.entry = nentries + ci;
            emask.push_back(s);
            ents.push_back(Entry{s, sb.comp, sb.csize, sb.inres, memP + (size_t) ci * n, 0, 0});
            ++ci;
        }
        for (size_t u = 0; u < stamps.size(); ++u) {
            stamps[u].dst = stamp_of[stamp_b[u]];
            copies.push_back(stamps[u]);
        }
        X.rootpos = batch.take<int>((size_t) ncomp * n + 4);  // the grouped link walk reads up to 3 past a run
        X.par = batch.take<int>((size_t) ncomp * n);
        X.giant = batch.take<int>(ncomp);
        X.fit = batch.take<int>(ncomp);
        if (fan) index_of(hc, ctab2);
    }
    std::vector<int> cb(copies.size() + 1, 0);
    for (size_t c = 0; c < copies.size(); ++c) cb[c + 1] = cb[c] + nblocks(copies[c].len);
    defer_uploads();
    PruneChild *dpc = nprune ? upload(batch, prune) : nullptr;
    int *dbw = nprune ? upload(batch, bw) : nullptr;
    int *dbp = nprune ? upload(batch, bp) : nullptr;
    if (any_chains) upload_chains(chains);
    CopySeg *dcs = copies.empty() ? nullptr : upload(batch, copies);
    int *dcb2 = copies.empty() ? nullptr : upload(batch, cb);
    if (ncomp > 0 && fan) columns(hc, ctab2);
    BatchSub *dhc = ncomp > 0 ? upload(batch, hc) : nullptr;
    if (ncomp > 0) put(entries + nentries, ents.data(), ents.size() * sizeof(Entry));
    flush_uploads();
    HIP_OK(launch_fill_many(post, st));
    if (any_chains) prune_chains(chains);
    if (nprune) HIP_OK(launch_b_prune(D, dpc, nprune, dbw, bw[nprune], dbp, bp[nprune], st));
    if (!copies.empty()) HIP_OK(launch_b_copy(dcs, dcb2, (int) copies.size(), cb.back(), st));
    if (ncomp > 0) {
        std::chrono::steady_clock::time_point tc0, tc1, tc2;
        if (dbg) {
            sync();
            tc0 = std::chrono::steady_clock::now();
        }
        HIP_OK(launch_b_count(dhc, ncomp, nullptr, 0, n, k, kfast, X, s_star, prm.neighborhood_size, phi_mode, phi_all_exact, D,
                              rank_perm, small + kStatAt, timer(), st));
        if (dbg) {
            sync();
            tc1 = std::chrono::steady_clock::now();
        }
        HIP_OK(launch_b_components(dhc, ncomp, n, k, kfast, X, s_star, st));
        if (dbg) {
            sync();
            tc2 = std::chrono::steady_clock::now();
            long long qs = 0;
            for (const BatchSub &x : ws) qs += x.qmax;
            auto ms = [](std::chrono::steady_clock::time_point a, std::chrono::steady_clock::time_point b) {
                return std::chrono::duration<double, std::milli>(b - a).count();
            };
            std::fprintf(stderr,
                         "[inscy batch] B=%d walked=%d k=%d cap=%d queries<=%lld list_count=%.3fms "
                         "comp=%d all_count=%.3fms components=%.3fms\n",
                         B, nw, k, cap_of(k), qs, ms(tq0, tq1), ncomp, ms(tc0, tc1), ms(tc1, tc2));
        }
        nentries += ncomp;
        stats.components += ncomp;
    }
}

// The restriction of a tree of mask s on dimension m, permuted level order.
PermStep Engine::perm_step(dmask_t s, int m) const {
    PermStep p;
    std::memset(&p, 0, sizeof(p));
    p.m = m;
    p.Lm = lvl_of[m];
    p.tree = levels_of(s);
    p.restricted = p.tree | dbit(p.Lm);
    p.tkey = -1;
    bool deeper = false, kept_below = false;
    for (int t = d - 1; t >= 0; --t) {
        if (dhas(p.restricted, t)) continue;
        if (level[t] > m) p.big |= dbit(t);
        if (t > p.Lm) {
            deeper = true;
        } else {
            if (p.tkey < 0) p.tkey = t;
            kept_below |= level[t] > m;
            if (kept_below) p.cond |= dbit(t);
        }
    }
    // m's level the deepest free one, and none above it or a larger dimension's
    p.filt = !deeper && (p.tkey < 0 || level[p.tkey] > m);
    return p;
}

// The subspaces S minus one dimension whose counts are complete (their
// dense components were built) bound the counts of S from above; a bound
// decides a point only below both thresholds of S and below the cap of the
// smaller subspaces, under which their counts are exact.
void Engine::set_bounds(dmask_t s, BatchSub &x) {
    const int k = x.S.k;
    int lo = std::min(weak_thr, dense_thr[k]);
    x.nbound = 0;
    x.lo = lo;
    for (int t = 0; t < k && x.nbound < kMaxBounds; ++t) {
        const dmask_t sub = s & ~dbit(x.S.dims[t]);
        auto it = subs.find(sub);
        if (!sub || it == subs.end() || it->second.entry < 0) continue;
        if (permuted) {
            // the cells of a dimension that only S minus t matches do not
            // restrict the neighbours in S
            const SubspaceArg Q = arg_of(sub);
            uint64_t mq = match_of(Q), ms = match_of(x.S);
            bool inside = true;
            for (int u = 0; u < Q.k; ++u)
                if ((mq >> u) & 1) inside &= (ms >> (u < t ? u : u + 1)) & 1;
            if (!inside) continue;
        }
        x.bound[x.nbound++] = it->second.cnt;
    }
    // counts are exact below the cap of |S| - 1 (phi: the stored values carry
    // an upper bound, used in the kernel)
    if (x.nbound > 0 && !phi_mode) lo = std::min(lo, cap_of(k - 1));
    x.lo = lo;
}

// pruneRedundancy and join, replayed in stages.  The reference's order visits
// per dimension every surviving child's subtree, then its pruneRedundancy,
// then the join of the kept children's clusters.  A step on subspace S reads
// the result rows of the supersets of S and writes the row of S, so two steps
// must keep their order exactly when one subspace contains the other; each
// step goes to the stage after the last earlier step it depends on, and the
// steps of one stage run together, a handful of launches per stage.
void Engine::replay_staged() {
    struct Step {
        dmask_t s;
        int kind, tree, t_lo, t_hi;
    };
    std::vector<Step> steps;
    std::vector<int> pass;
    std::function<void(int)> walk = [&](int f) {
        const std::vector<int> &kids = lt[f].kids;
        size_t i = 0;
        while (i < kids.size()) {
            const int m = lt[kids[i]].m;
            size_t j = i;
            int t_lo = INT_MAX, t_hi = -1;
            std::vector<int> pk;
            while (j < kids.size() && lt[kids[j]].m == m) {
                t_lo = std::min(t_lo, kids[j]);
                t_hi = std::max(t_hi, kids[j] + 1);
                if (lt[kids[j]].pass) pk.push_back(kids[j]);
                ++j;
            }
            const dmask_t s = lt[kids[i]].smask;
            if (pk.size() == 1) {
                walk(pk[0]);
                steps.push_back({s, 0, pk[0], pk[0], pk[0] + 1});
            } else if (!pk.empty()) {
                for (int c : pk) {
                    walk(c);
                    steps.push_back({s, 1, c, c, c + 1});
                }
                steps.push_back({s, 2, -1, t_lo, t_hi});
            }
            i = j;
        }
    };
    walk(0);
    // stages: last_on[r] = last stage of a step on row r, last_sub[r] = last
    // stage of a step on a subspace of row r
    const int ne = (int) emask.size();
    std::vector<int> last_on(ne, 0), last_sub(ne, 0), stage(steps.size());
    int nst = 0;
    for (size_t i = 0; i < steps.size(); ++i) {
        const Subspace &sb = subs.at(steps[i].s);
        const auto sl = sup_at.at(steps[i].s);
        int st0 = last_sub[sb.entry];
        for (int u = 0; u < sl.second; ++u) st0 = std::max(st0, last_on[sup_flat[sl.first + u]]);
        const int sti = st0 + 1;
        stage[i] = sti;
        nst = std::max(nst, sti);
        last_on[sb.entry] = std::max(last_on[sb.entry], sti);
        for (int u = 0; u < sl.second; ++u) {
            int &x = last_sub[sup_flat[sl.first + u]];
            x = std::max(x, sti);
        }
    }
    std::vector<std::vector<int>> by_stage(nst + 1);
    for (size_t i = 0; i < steps.size(); ++i) by_stage[stage[i]].push_back((int) i);
    if (batch_trace)
        std::fprintf(stderr, "[inscy replay] %zu steps in %d stages\n", steps.size(), nst);

    // per step: row flags (2 per superset row) and a block counter
    // (redundancy), the join's two words and its candidate list
    const size_t kScratchInts = (size_t) 64 << 20;  // per launch group
    batch.reset();
    size_t held = 0;  // scratch of the chunks in flight
    const int ccap = prm.min_size > 0 ? std::min(n, n / prm.min_size + 1) : n;
    for (int sg = 1; sg <= nst; ++sg) {
        const std::vector<int> &ids = by_stage[sg];
        size_t a = 0;
        while (a < ids.size()) {
            // a chunk of the stage whose scratch fits the budget
            size_t b = a, ints = 0;
            while (b < ids.size()) {
                const Step &x = steps[ids[b]];
                const size_t need = 2 * (size_t) sup_at.at(x.s).second + 3 + (x.kind == 1 ? 0 : (size_t) ccap);
                if (b > a && ints + need > kScratchInts) break;
                ints += need;
                ++b;
            }
            if (held > 0 && held + ints > kScratchInts) {
                sync();  // the chunks in flight still use theirs
                batch.reset();
                held = 0;
            }
            held += ints + 65536;  // with its descriptors
            int *scr = batch.take<int>(std::max<size_t>(ints, 1));
            HIP_OK(launch_fill_i32(scr, 0, std::max<size_t>(ints, 1), st));
            std::vector<RepOp> ops(b - a);
            std::vector<int> br{0}, bc{0}, bk{0}, bm{0};
            size_t at = 0;
            for (size_t u = a; u < b; ++u) {
                const Step &x = steps[ids[u]];
                const Subspace &sb = subs.at(x.s);
                const auto sl = sup_at.at(x.s);
                RepOp &o = ops[u - a];
                std::memset(&o, 0, sizeof(o));
                o.list = d_sup + sl.first;
                o.nlist = sl.second;
                o.tstamp = sb.tstamp;
                o.flag = sb.cnt;
                o.comp = sb.comp;
                o.csize = sb.csize;
                o.inres = sb.inres;
                o.entry = sb.entry;
                o.kind = x.kind;
                o.tree = x.tree;
                o.t_lo = x.t_lo;
                o.t_hi = x.t_hi;
                o.J = x.kind == 1 ? 0 : ++rep_join;
                o.ccap = ccap;
                o.rowflag = scr + at;
                at += 2 * (size_t) sl.second;
                o.done = reinterpret_cast<unsigned *>(scr + at);
                at += 1;
                o.words = scr + at;
                at += 2;
                if (x.kind != 1) {
                    o.clist = scr + at;
                    at += ccap;
                }
                if (x.tree >= 0) {
                    o.W = lt[x.tree].W;
                    o.nW = lt[x.tree].nW;
                }
                br.push_back(br.back() + (x.kind != 2 ? rep_red_blocks(o.nlist, o.nW) : 0));
                bc.push_back(bc.back() + (x.kind == 0 ? (int) std::max(1u, blocks_for_host(o.nW))
                                                      : x.kind == 2 ? (int) blocks_for_host(n) : 0));
                bk.push_back(bk.back() + (x.kind != 1 ? rep_check_blocks(o.nlist, n) : 0));
                bm.push_back(bm.back() + (x.kind != 1 ? rep_mem_blocks(n) : 0));
            }
            const int no = (int) ops.size();
            defer_uploads();
            RepOp *dops = upload(batch, ops);
            int *dbr = upload(batch, br), *dbc = upload(batch, bc), *dbk = upload(batch, bk), *dbm = upload(batch, bm);
            flush_uploads();
            HIP_OK(launch_rep_stage(dops, no, dbr, br.back(), dbc, bc.back(), dbk, bk.back(), dbm, bm.back(), entries,
                                    prm.r, prm.min_size, n, keepv, st));
            a = b;
        }
    }
}

// Features of every (tree, dimension) pair of the level (learned and collect
// modes) and, with a pruner loaded, its decisions: a pair whose score is below
// the threshold is skipped, unless its tree has fewer than prune_min_depth
// restricted dimensions.
void Engine::score_pairs(int na) {
    Pool &cur = lvl[cur_lvl];
    lv_pair0.assign(na, 0);
    std::vector<FeatPair> fp;
    std::vector<int> blk{0};
    for (int a = 0; a < na; ++a) {
        const LTree &t = lt[lv_act[a]];
        lv_pair0[a] = (int) fp.size();
        // counts of S are complete for every subspace holding a surviving
        // tree; in phi mode they are decision bits and are left out
        const int *cntS = t.smask && !phi_mode ? subs.at(t.smask).cnt : nullptr;
        const int k = dcount(t.smask);
        for (int m = t.first; m < d; ++m) {
            FeatPair f;
            std::memset(&f, 0, sizeof(f));
            f.W = t.W;
            f.cntS = cntS;
            f.gid = lv_gid + lv_gidoff[a] + (m - t.first) * cells;
            f.mask = t.smask | dbit(m);
            f.nW = t.nW;
            f.pre = t.pre;
            f.m = m;
            f.k = k;
            f.first = t.first;
            f.ngroups = (int) lv_groups[a][m - t.first].size();
            f.bp = nblocks(t.nW);
            f.cap = cap_of(k);
            fp.push_back(f);
            blk.push_back(blk.back() + f.bp);
        }
    }
    const int np = (int) fp.size();
    stats.pairs_scored += np;
    if (np == 0) return;
    const size_t stride = (size_t) kHistBins + cells + 2;
    int *acc = cur.take<int>((size_t) np * stride);
    unsigned long long *accs = cur.take<unsigned long long>(np);
    float *feat = cur.take<float>((size_t) np * kMlpIn);
    HIP_OK(launch_fill_i32(acc, 0, (size_t) np * stride, st));
    HIP_OK(launch_fill_u64(reinterpret_cast<uint64_t *>(accs), 0ull, np, st));
    defer_uploads();
    FeatPair *dfp = upload(cur, fp);
    int *dblk = upload(cur, blk);
    flush_uploads();
    HIP_OK(launch_pair_features(dfp, dblk, np, blk[np], D.Xt, cellC, n, d, cells, prm.min_size, weak_thr, acc, accs,
                                feat, st));
    if (collect) {
        col_base = (long long) col_tree.size();
        const size_t at = col_feat.size();
        col_feat.resize(at + (size_t) np * kMlpIn);
        float *h = reinterpret_cast<float *>(down.get((size_t) np * kMlpIn * sizeof(float)));
        HIP_OK(hipMemcpyAsync(h, feat, (size_t) np * kMlpIn * sizeof(float), hipMemcpyDeviceToHost, st));
        sync();
        std::memcpy(col_feat.data() + at, h, (size_t) np * kMlpIn * sizeof(float));
        for (int a = 0; a < na; ++a)
            for (int m = lt[lv_act[a]].first; m < d; ++m) {
                col_tree.push_back(lv_act[a]);
                col_m.push_back(m);
                col_child0.push_back(-1);
                col_G.push_back(0);
            }
    }
    if (pruner) {
        float *prob = cur.take<float>(np);
        HIP_OK(launch_mlp_predict(feat, np, pruner, prob, st));
        const float *hp = reinterpret_cast<const float *>(down.get((size_t) np * sizeof(float)));
        HIP_OK(hipMemcpyAsync(const_cast<float *>(hp), prob, (size_t) np * sizeof(float), hipMemcpyDeviceToHost, st));
        sync();
        lv_skip.assign(np, 0);
        for (int a = 0; a < na; ++a) {
            const LTree &t = lt[lv_act[a]];
            if (dcount(t.smask) < prune_min_depth) continue;
            for (int m = t.first; m < d; ++m) {
                const int j = lv_pair0[a] + m - t.first;
                if (hp[j] < prune_thr) {
                    lv_skip[j] = 1;
                    stats.pairs_skipped++;
                }
            }
        }
    }
}

// Labels of the collected pairs.  A surviving tree holds a result cluster
// when it was kept by pruneRedundancy and one of its points lies in a cluster
// of the result in its subspace; a pair is positive when a tree below it (a
// child along its dimension, or any descendant of one) holds a result cluster.
void Engine::finish_collect(inscy_result &out) {
    const int nt = (int) lt.size();
    std::vector<TreeHit> th;
    std::vector<int> blk{0};
    for (int i = 1; i < nt; ++i) {
        const LTree &t = lt[i];
        if (!t.pass || t.nW <= 0) continue;
        const Subspace &sb = subs.at(t.smask);
        th.push_back(TreeHit{t.W, sb.comp, sb.inres, t.nW, i});
        blk.push_back(blk.back() + nblocks(t.nW));
    }
    int *hit = store.take<int>(std::max(nt, 1));
    HIP_OK(launch_fill_i32(hit, 0, std::max(nt, 1), st));
    if (!th.empty()) {
        defer_uploads();
        TreeHit *dth = upload(store, th);
        int *dblk = upload(store, blk);
        flush_uploads();
        HIP_OK(launch_tree_hits(dth, dblk, (int) th.size(), blk.back(), hit, st));
    }
    std::vector<int> hh(nt), keep(nt);
    HIP_OK(hipMemcpyAsync(hh.data(), hit, (size_t) nt * sizeof(int), hipMemcpyDeviceToHost, st));
    HIP_OK(hipMemcpyAsync(keep.data(), keepv, (size_t) nt * sizeof(int), hipMemcpyDeviceToHost, st));
    sync();
    const long long np = (long long) col_tree.size();
    // pairs of each tree (contiguous in collection order)
    std::vector<long long> p0(nt, -1), pn(nt, 0);
    for (long long j = 0; j < np; ++j) {
        if (p0[col_tree[j]] < 0) p0[col_tree[j]] = j;
        pn[col_tree[j]]++;
    }
    // children have larger indices than their parents
    std::vector<char> contrib(nt, 0);
    std::vector<long long> tcost(nt, 0);
    out.pair_label.assign(np, 0);
    out.pair_cost.assign(2 * np, 0);
    out.pair_info.assign(4 * np, 0);
    for (int i = nt - 1; i >= 0; --i) {
        const LTree &t = lt[i];
        bool c = i > 0 && t.pass && keep[i] && hh[i];
        long long tc = 0;
        for (long long j = p0[i]; j >= 0 && j < p0[i] + pn[i]; ++j) {
            bool pos = false;
            long long cost = t.nW;
            for (int u = 0; u < col_G[j]; ++u) {
                const int ch = col_child0[j] + u;
                pos |= contrib[ch] != 0;
                cost += tcost[ch];
            }
            out.pair_label[j] = pos ? 1 : 0;
            out.pair_cost[2 * j] = t.nW;
            out.pair_cost[2 * j + 1] = cost;
            out.pair_info[4 * j] = dcount(t.smask);
            out.pair_info[4 * j + 1] = col_m[j];
            out.pair_info[4 * j + 2] = t.nW;
            out.pair_info[4 * j + 3] = i;
            c |= pos;
            tc += cost;
        }
        contrib[i] = c;
        tcost[i] = tc;
    }
    out.pair_feat = std::move(col_feat);
    col_feat.clear();
}

void Engine::trace_tree(int f, const std::vector<int> &keep) {
    for (int c : lt[f].kids) {
        const LTree &t = lt[c];
        trace.push_back({(long long) dlo(t.smask), t.lo, t.hi, t.pre, t.nW, t.pass ? 1 : 0,
                         t.pass ? (keep[c] ? 0 : 1) : -1});
        if (t.pass) trace_tree(c, keep);
    }
}

}  // namespace inscy
