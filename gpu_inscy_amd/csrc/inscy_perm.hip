// Permuted SCY-tree level order (entropy_order != 0, get_subspace_order,
// inscy_map.cpp:61-121): the tree passes of the level-synchronous driver over
// s-connection chains.
//
// With the levels in a permuted order, restrict_node (ScyTreeNode.cu:227-320)
// keeps every node whose dimension id exceeds the restricted one, so a
// restricted tree holds empty regular nodes and truncated s-connection chains,
// and mergeNodes (ScyTreeNode.cu:803-833) adds counts and points only into
// nodes whose count is positive.  A tree here is its points P (the weak-dense
// points of its last prune) and its chains: (x, b, end) is the chain point x
// starts at the level of dimension b, running through x's cells down to level
// `end` (restricted levels skipped).  Per restriction on m and cell group G:
//  - merge flags: chains with b == m, by x's cell in m;
//  - points: those with their cell in G; when m's level is the deepest
//    unrestricted one and the level above it has a dimension id above m (or
//    none is left), only prefixes holding a point of G's first cell keep
//    theirs (the tree of that cell has an empty node there, which mergeNodes
//    does not add to);
//  - chains (b != m): a chain below m's level is reached only through x's
//    cell and keeps its nodes down to the deepest one with dimension id above
//    m; a chain above passes when its cell is in G (keeping the part below
//    down to the deepest such node, else ending just above m's level), and
//    otherwise keeps its nodes down to the deepest one above m's level with a
//    dimension id above m;
//  - prune (pruneRecursionAndRemove2 + propergate_count2): a chain stays when
//    its regular parent keeps a weak-dense point, unless its same-cell
//    regular sibling existed before the prune (a prefix of the tree's points,
//    an ancestor of one of its chains, or a node above m's level kept because
//    a level between it and m's has a dimension id above m) and lost its
//    weak-dense points.
// The prefixes that a child's prune asks about (two per routed chain: its parent
// and its sibling) go into an open-addressing table of (25 hash bits | level |
// point), every hit confirmed by comparing cells; the tree's points and chains
// look theirs up and mark the ones found.  Every pass serves all (tree,
// dimension) pairs or children of a batch in one launch: one tree at a time the
// launches were the bound (n=3,001 d=9: 4,666 launches and 26.5 ms a run, 166 and
// 2.0 ms in this form).
#include "inscy_internal.h"

#include "inscy_device.h"

namespace inscy {

namespace {

__device__ __forceinline__ int chain_b(uint64_t w) { return (int) (w & 0xFFull); }
__device__ __forceinline__ int chain_end(uint64_t w) { return (int) ((w >> 8) & 0xFFull); }
__device__ __forceinline__ uint64_t chain_word(int b, int end) { return (uint64_t) b | ((uint64_t) end << 8); }

constexpr uint64_t kSeed = 0x243F6A8885A308D3ull;
__device__ __forceinline__ uint64_t level_salt(int t) { return 0x9E3779B97F4A7C15ull * (uint64_t) (t + 1); }
// levels from..to (empty when to < from)
__device__ __forceinline__ dmask_t levels_in(int from, int to) { return dabove(from - 1) & ~dabove(to); }

// f(t, hash) for the prefix of z through every level t of `want` (unrestricted ones)
template <class F>
__device__ __forceinline__ void prefixes(const DevData &D, dmask_t restricted, int z, dmask_t want, F f) {
    uint64_t h = kSeed;
    CellRow row{};
    for (int t = 0; want && t < D.d; ++t) {
        if (!(t & 15)) row = load_row(D, z, t);
        if (dhas(restricted, t)) continue;
        h = mix64(h + row.at(t & 15) + 1);
        if (!dhas(want, t)) continue;
        want &= ~dbit(t);
        f(t, mix64(h ^ level_salt(t)));
    }
}

// a table entry: 25 hash bits | level | point (n < 2^30, so never kEmpty)
__device__ __forceinline__ uint64_t table_entry(uint64_t e, int z, int t) {
    return (e >> 39) << 39 | (uint64_t) t << 32 | (uint32_t) z;
}
// slot of the prefix e of z through level t, inserted when it is not there
// (insert false: -1 then); accept(point) decides beyond the cells
template <bool INSERT, class F>
__device__ __forceinline__ long long table_slot(const DevData &D, dmask_t restricted, uint64_t *table, uint64_t tmask,
                                                uint64_t e, int z, int t, F accept) {
    const uint64_t entry = table_entry(e, z, t);
    uint64_t slot = e & tmask;
    while (true) {
        // a slot is written once, by the swap from empty: a plain load that
        // still sees it empty is corrected by the failed swap, a full one is final
        uint64_t cur = table[slot];
        if (cur == kEmpty) {
            if (!INSERT) return -1;
            cur = atomicCAS((unsigned long long *) &table[slot], (unsigned long long) kEmpty,
                            (unsigned long long) entry);
            if (cur == kEmpty) return (long long) slot;
        }
        if ((cur >> 32) == (entry >> 32) && accept((int) (uint32_t) cur) &&
            same_prefix(D, restricted, z, (int) (uint32_t) cur, t))
            return (long long) slot;
        slot = (slot + 1) & tmask;
    }
}
struct AnyPoint {
    __device__ __forceinline__ bool operator()(int) const { return true; }
};

// the root tree: every point, a chain to the deepest level for every near-edge
// dimension of a point; and the cell edges
__global__ void k_p_root(const dmask_t *__restrict__ nearm, int n, int d, int *__restrict__ P, int *__restrict__ cx,
                         uint64_t *__restrict__ cw, int *__restrict__ nout, int C, float *__restrict__ edge) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < C + 3) edge[i] = cell_edge(i, C);
    if (i < n) P[i] = i;
    dmask_t m = i < n ? nearm[i] : (dmask_t) 0;
    const int lane = __lane_id();
    int at = dcount(m);
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(at, o);
        if (lane >= o) at += v;
    }
    int base = 0;
    if (lane == 63 && at) base = atomicAdd(nout, at);
    at += __shfl(base, 63) - dcount(m);
    while (m) {
        const int b = dfirst(m);
        m &= m - 1;
        cx[at] = i;
        cw[at++] = chain_word(b, d - 1);
    }
}

__global__ void k_p_chains(const dmask_t *__restrict__ nearm, int n, unsigned long long *__restrict__ total) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    int c = i < n ? dcount(nearm[i]) : 0;
    for (int o = 32; o > 0; o >>= 1) c += __shfl_down(c, o);
    if (__lane_id() == 0 && c) atomicAdd(total, (unsigned long long) c);
}

// merge flags of every dimension >= first of every tree
__global__ void k_p_flags(const FlagTree *__restrict__ T, const int *__restrict__ blk_off, int nt,
                          const uint8_t *__restrict__ cellC, int n, int cells, int *__restrict__ flags) {
    const int t = seg_of(blk_off, nt, blockIdx.x);
    const FlagTree F = T[t];
    const int i = (blockIdx.x - blk_off[t]) * blockDim.x + threadIdx.x;
    if (i >= *F.nsp) return;
    const int b = chain_b(F.spm[i]);
    if (b < F.first) return;
    flags[F.flag_off + (b - F.first) * cells + cellC[(size_t) b * n + F.spx[i]]] = 1;
}

// end of a chain after the step, in the group of x's cell (in) or in another
// one; -1 where the chain does not pass
__device__ __forceinline__ int route(const PermStep &s, int Lb, int end, bool in) {
    if (Lb > s.Lm) return in ? dlast(s.big & levels_in(Lb, end)) : -1;
    if (end >= s.Lm && in) {
        const int e = dlast(s.big & levels_in(s.Lm + 1, end));
        // else the chain node above the restricted level
        return e >= 0 ? e : max(Lb, dlast(~s.tree & levels_in(Lb, s.Lm - 1)));
    }
    return dlast(s.big & levels_in(Lb, min(end, s.Lm - 1)));
}

// how many chains of every pair go to each of its groups
__global__ void k_p_count(DevData D, const PermPair *__restrict__ pairs, const int *__restrict__ blk_off, int np) {
    __shared__ int h[2 * 256];
    const int j = seg_of(blk_off, np, blockIdx.x);
    const PermPair &A = pairs[j];
    const int G = A.G;
    for (int t = threadIdx.x; t < 2 * G; t += blockDim.x) h[t] = 0;
    __syncthreads();
    const int i = (blockIdx.x - blk_off[j]) * blockDim.x + threadIdx.x;
    if (i < A.nsp) {
        const uint64_t w = A.chain[i];
        const int b = chain_b(w), end = chain_end(w);
        if (b != A.s.m) {
            const int Lb = D.lvl_of[b], g = A.gid[D.cellC[(size_t) A.s.m * D.n + A.spx[i]]];
            if (route(A.s, Lb, end, true) >= 0) atomicAdd(&h[g], 1);
            if (route(A.s, Lb, end, false) >= 0) atomicAdd(&h[G + g], 1);
        }
    }
    __syncthreads();
    for (int t = threadIdx.x; t < 2 * G; t += blockDim.x)
        if (h[t]) atomicAdd(t < G ? &A.in[t] : &A.out[t - G], h[t]);
}

// The points of every group's first cell enter their prefixes (through the
// deepest free level above m's), then every point looks its own up among its
// group's.
template <bool MARK>
__global__ void k_p_filter(DevData D, const PermFilter *__restrict__ filters, const int *__restrict__ blk_off, int nf) {
    const int j = seg_of(blk_off, nf, blockIdx.x);
    const PermFilter &F = filters[j];
    const int i = (blockIdx.x - blk_off[j]) * blockDim.x + threadIdx.x;
    if (i >= F.nP) return;
    const int z = F.P[i];
    const uint8_t *cm = D.cellC + (size_t) F.s.m * D.n;
    const int c = cm[z], g = F.gid[c];
    const bool lo = c == 0 || F.gid[c - 1] != g;
    if (MARK && !lo) return;
    bool found = lo;
    if (MARK || !lo) {
        const int tk = F.s.tkey;
        uint64_t e = kSeed;
        if (tk >= 0) prefixes(D, F.s.restricted, z, dbit(tk), [&](int, uint64_t h) { e = h; });
        e = mix64(e + (uint64_t) g);
        found = table_slot<MARK>(D, F.s.restricted, F.table, F.tmask, e, z, tk < 0 ? 0 : tk, [&](int y) {
                    return y >= 0 && y < D.n && F.gid[cm[y]] == g;
                }) >= 0;
    }
    if (!MARK) F.keep[i] = found;
}

// a child's chains out of its parent's, and the prefixes its prune asks about:
// x's through the last free level above b's (the chain's regular parent) and
// through b's (its regular sibling)
__global__ void k_p_route(DevData D, const PermChild *__restrict__ C, const int *__restrict__ blk_off, int nc) {
    const int c = seg_of(blk_off, nc, blockIdx.x);
    const PermChild &P = C[c];
    const int i = (blockIdx.x - blk_off[c]) * blockDim.x + threadIdx.x;
    int x = 0, b = 0, e = -1, Lb = 0;
    if (i < P.nsp) {
        const uint64_t w = P.chain[i];
        b = chain_b(w);
        x = P.spx[i];
        if (b != P.s.m) {
            Lb = D.lvl_of[b];
            e = route(P.s, Lb, chain_end(w), P.gid[D.cellC[(size_t) P.s.m * D.n + x]] == P.g);
        }
    }
    const int at = wave_slot(e >= 0, P.nr_at);
    dmask_t want = 0;
    if (e >= 0) {
        P.rx[at] = x;
        P.rw[at] = chain_word(b, e);
        const int tp = dlast(~P.s.restricted & levels_in(0, Lb - 1));
        want = dbit(Lb) | (tp >= 0 ? dbit(tp) : (dmask_t) 0);
    }
    wave_or_mask(want, P.bits);
    if (!want) return;
    prefixes(D, P.s.restricted, x, want, [&](int t, uint64_t h) {
        table_slot<true>(D, P.s.restricted, P.table, P.tmask, h, x, t, AnyPoint{});
    });
}

// Marks of the prefixes asked for.  The parent's points: in the child, the node
// existed and, weak-dense, still holds a point; elsewhere it existed at the
// levels of `cond`.  Then the routed chains: their regular ancestors existed.
__global__ void k_p_mark(DevData D, const PermChild *__restrict__ C, const int *__restrict__ blk_off, int nc, int thr,
                         int wbit) {
    const int c = seg_of(blk_off, nc, blockIdx.x);
    const PermChild &P = C[c];
    const int i = (blockIdx.x - blk_off[c]) * blockDim.x + threadIdx.x;
    const dmask_t need = *P.bits;
    dmask_t exist = 0;
    int z = 0;
    bool weak = false;
    if (i < P.nP) {
        z = P.P[i];
        if (P.gid[D.cellC[(size_t) P.s.m * D.n + z]] == P.g && (!P.keep || P.keep[i])) {
            exist = need;
            weak = meets(P.weakcnt[z], thr, wbit);
        } else {
            exist = need & P.s.cond;
        }
    } else if (i < P.nP + P.nr) {
        z = P.rx[i - P.nP];
        exist = need & levels_in(0, D.lvl_of[chain_b(P.rw[i - P.nP])] - 1);
    }
    prefixes(D, P.s.restricted, z, exist, [&](int t, uint64_t h) {
        const long long at = table_slot<false>(D, P.s.restricted, P.table, P.tmask, h, z, t, AnyPoint{});
        if (at < 0) return;
        // every marker writes the same byte
        if (weak && !P.marks[2 * at]) P.marks[2 * at] = 1;
        if (!P.marks[2 * at + 1]) P.marks[2 * at + 1] = 1;
    });
}

__global__ void k_p_check(DevData D, const PermChild *__restrict__ C, const int *__restrict__ blk_off, int nc) {
    const int c = seg_of(blk_off, nc, blockIdx.x);
    const PermChild &P = C[c];
    const int i = (blockIdx.x - blk_off[c]) * blockDim.x + threadIdx.x;
    int x = 0;
    uint64_t w = 0;
    bool keep = false;
    if (i < P.nr) {
        x = P.rx[i];
        w = P.rw[i];
        const int Lb = D.lvl_of[chain_b(w)];
        const int tp = dlast(~P.s.restricted & levels_in(0, Lb - 1));
        keep = true;
        prefixes(D, P.s.restricted, x, dbit(Lb) | (tp >= 0 ? dbit(tp) : (dmask_t) 0), [&](int t, uint64_t h) {
            const long long at = table_slot<false>(D, P.s.restricted, P.table, P.tmask, h, x, t, AnyPoint{});
            const bool holds = at >= 0 && P.marks[2 * at], was = at >= 0 && P.marks[2 * at + 1];
            // the parent holds no point, or the sibling lost its points
            // (propergate_count2 erases the chain)
            if (!holds && (t != Lb || was)) keep = false;
        });
    }
    const int at = wave_slot(keep, P.nout);
    if (keep) {
        P.outx[at] = x;
        P.outw[at] = w;
    }
}

}  // namespace

#define LAUNCH(kernel, grid, block, lds, st, ...) hipLaunchKernelGGL(kernel, grid, block, lds, st, __VA_ARGS__)

hipError_t launch_p_root(const dmask_t *nearm, int n, int d, int *P, int *cx, uint64_t *cw, int *nout, int C,
                         float *edge, hipStream_t st) {
    LAUNCH(k_p_root, dim3(blocks_for((size_t) std::max(n, C + 3))), dim3(kBlock), 0, st, nearm, n, d, P, cx, cw, nout, C,
           edge);
    return hipGetLastError();
}

hipError_t launch_p_chains(const dmask_t *nearm, int n, unsigned long long *total, hipStream_t st) {
    LAUNCH(k_p_chains, dim3(blocks_for(n)), dim3(kBlock), 0, st, nearm, n, total);
    return hipGetLastError();
}

hipError_t launch_p_flags(const FlagTree *T, const int *blk_off, int nt, int nblk, const uint8_t *cellC, int n,
                          int cells, int *flags, hipStream_t st) {
    if (nblk <= 0) return hipSuccess;
    LAUNCH(k_p_flags, dim3(nblk), dim3(kBlock), 0, st, T, blk_off, nt, cellC, n, cells, flags);
    return hipGetLastError();
}

hipError_t launch_p_filter(const DevData &D, const PermFilter *F, const int *blk_off, int nf, int nblk,
                           hipStream_t st) {
    if (nblk <= 0) return hipSuccess;
    LAUNCH(k_p_filter<true>, dim3(nblk), dim3(kBlock), 0, st, D, F, blk_off, nf);
    LAUNCH(k_p_filter<false>, dim3(nblk), dim3(kBlock), 0, st, D, F, blk_off, nf);
    return hipGetLastError();
}

hipError_t launch_p_count(const DevData &D, const PermPair *P, const int *blk_off, int np, int nblk, hipStream_t st) {
    if (nblk <= 0) return hipSuccess;
    LAUNCH(k_p_count, dim3(nblk), dim3(kBlock), 0, st, D, P, blk_off, np);
    return hipGetLastError();
}

hipError_t launch_p_prune(const DevData &D, const PermChild *C, int nc, const int *blk_route, int nblk_route,
                          const int *blk_mark, int nblk_mark, const int *blk_check, int nblk_check, int thr, int wbit,
                          hipStream_t st) {
    if (nc <= 0) return hipSuccess;
    if (nblk_route > 0) LAUNCH(k_p_route, dim3(nblk_route), dim3(kBlock), 0, st, D, C, blk_route, nc);
    if (nblk_mark > 0) LAUNCH(k_p_mark, dim3(nblk_mark), dim3(kBlock), 0, st, D, C, blk_mark, nc, thr, wbit);
    if (nblk_check > 0) LAUNCH(k_p_check, dim3(nblk_check), dim3(kBlock), 0, st, D, C, blk_check, nc);
    return hipGetLastError();
}

}  // namespace inscy
