// Level-synchronous passes of the MI355X INSCY engine (gfx950, wave64).
//
// Every launch covers a whole batch: all trees of one
// recursion level (merge flags, partition, path prune) or many subspaces (grid
// index, neighbour counts, dense components).  A block belongs to exactly one
// segment, found by a binary search of its block offsets, so a wave never
// mixes segments and the wave-aggregated compaction stays valid.
//
// Floating point follows inscy_kernels.hip: no contraction, and the distance
// test is sum <= s_star.

#include <algorithm>
#include <climits>


#include "inscy_device.h"
#include "inscy_internal.h"

#pragma clang fp contract(off)

namespace inscy {

namespace {

constexpr int kBLanes = 4;  // lanes per query of the batched neighbour passes (one quad: the walks sum over it with DPP)
constexpr int QPB = kBlock / kBLanes;
static_assert(kBLanes == 4, "the walks' tally sums a query's lanes as one DPP quad");
static_assert(QPB == kQueriesPerBlock, "queries per block of the host and the kernels");

__device__ __forceinline__ int origin(int x) { return x >= 0 ? x : ~x; }

// ------------------------------------------------------------ merge flags of every tree of a level
// (ScyTreeNode.cu:837-851 with restrict_node :262-267)
__global__ void k_b_flags(const FlagTree *__restrict__ T, const int *__restrict__ blk_off, int nt,
                          const uint8_t *__restrict__ cellC, int n, int cells, int *__restrict__ flags) {
    const int t = seg_of(blk_off, nt, blockIdx.x);
    const FlagTree F = T[t];
    const int i = (blockIdx.x - blk_off[t]) * blockDim.x + threadIdx.x;
    if (i >= *F.nsp) return;
    const int x = origin(F.spx[i]);
    dmask_t m = mload(F.spm, i, F.mw) & dabove(F.first - 1);
    int *fl = flags + F.flag_off;
    while (m) {
        const int b = dfirst(m);
        m &= m - 1;
        fl[(b - F.first) * cells + cellC[(size_t) b * n + x]] = 1;
    }
}

// the root tree: every point, the path of every point with a near-edge
// dimension; and the cell edges
__global__ void k_b_root(const dmask_t *__restrict__ nearm, int n, int *__restrict__ P, int *__restrict__ outx,
                         uint64_t *__restrict__ outm, int mw, int *__restrict__ nout, int C, float *__restrict__ edge) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < C + 3) edge[i] = cell_edge(i, C);
    if (i < n) P[i] = i;
    const dmask_t m = i < n ? nearm[i] : (dmask_t) 0;
    const int slot = wave_slot(m != 0, nout);
    if (m != 0) {
        outx[slot] = i;
        mstore(outm, slot, m, mw);
    }
}

// ------------------------------------------------------------ grid indexes of a batch of subspaces
// grid keys and in-cell ranks (grid.y = index); one counting sort per index
__global__ void k_b_keys(DevData D, const SortJob *__restrict__ jobs, int *__restrict__ keys, int *__restrict__ rank,
                         int *__restrict__ hist) {
    const SortJob &J = jobs[blockIdx.y];
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= D.n) return;
    int key = 0;
    const int jl = J.j - 1;
    for (int a = 0; a < jl; ++a) key = key * J.C + D.cellE[(size_t) J.dims[a] * D.n + p];
    // the last index dimension: its cell, or its bucket within the cell
    const int dl = J.dims[jl];
    if (J.F > 1)
        key = key * (J.C * J.F) + fine_key(D.Xt[(size_t) dl * D.n + p], J.C, J.F);
    else
        key = key * J.C + D.cellE[(size_t) dl * D.n + p];
    const size_t at = (size_t) blockIdx.y * D.n + p;
    keys[at] = key;
    rank[at] = atomicAdd(&hist[J.hoff + key], 1);
}

// `off` is one exclusive scan over the grid cells of every index of the
// batch, so its positions are global: index u holds [u*n, (u+1)*n).  The
// scatter writes the sorted ids, each point's sorted position and the index's
// own cell offsets to where the index is kept.
__global__ void k_b_scatter(int n, const SortJob *__restrict__ jobs, const int *__restrict__ keys,
                            const int *__restrict__ rank, const int *__restrict__ off) {
    const SortJob &J = jobs[blockIdx.y];
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    const int base = (int) ((long long) blockIdx.y * n);
    if (p < n) {
        const size_t src = (size_t) blockIdx.y * n + p;
        const int at = off[J.hoff + keys[src]] + rank[src] - base;
        J.order[at] = p;
        J.pos[p] = at;
    }
    if (p <= J.ncell) J.off[p] = off[J.hoff + p] - base;
}

// coordinate columns in sorted order, four positions per thread
constexpr int kGatherItems = 4;
__global__ void k_b_gather(const ColJob *__restrict__ jobs, int n, int nblk) {
    const int job = blockIdx.x / nblk, blk = blockIdx.x - job * nblk;
    const ColJob J = jobs[job];
    const int i0 = blk * kBlock * kGatherItems + threadIdx.x;
    int p[kGatherItems];
    float v[kGatherItems];
#pragma unroll
    for (int u = 0; u < kGatherItems; ++u) {
        const int i = i0 + u * kBlock;
        p[u] = i < n ? J.order[i] : 0;
    }
#pragma unroll
    for (int u = 0; u < kGatherItems; ++u) v[u] = J.src[p[u]];
#pragma unroll
    for (int u = 0; u < kGatherItems; ++u) {
        const int i = i0 + u * kBlock;
        if (i < n) J.dst[i] = v[u];
    }
}

// ------------------------------------------------------------ query lists in sorted order
__global__ void k_b_qmark(const BatchSub *__restrict__ subs, const QuerySeg *__restrict__ segs,
                          const int *__restrict__ blk_off, int nseg, uint8_t *__restrict__ qflag,
                          int *__restrict__ seg) {
    const int s = seg_of(blk_off, nseg, blockIdx.x);
    const QuerySeg Q = segs[s];
    const int i = (blockIdx.x - blk_off[s]) * blockDim.x + threadIdx.x;
    if (i >= Q.len) return;
    const BatchSub &B = subs[Q.b];
    const int p = Q.P[i];
    const long long at = B.base + B.pos[p];
    qflag[at] = 1;
    if (seg) seg[at] = s;
}

// ------------------------------------------------------------ candidate walk
// The candidates of a query are up to 9 runs of sorted positions (grid cells
// of the index dimensions).  They are concatenated into one index space
// [0, total): q[0..8] run starts (local positions), q[9..18] prefix sums of
// the run lengths (empty runs stay in place).  A lane maps its candidate
// number to a position with a run pointer that only moves forward.
// q[19]: the run of the query's own cells in the first index dimensions (it
// holds the query, so it is not empty).  q[20..29]: prefix sums of the runs'
// lengths in groups of four (ceil(length / 4)), for the walks that take four
// consecutive candidates of one run per lane.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// inclusive sum over the lanes of a quad (all four active)
__device__ __forceinline__ int quad_scan(int v, int sub) {
    int o = __builtin_amdgcn_update_dpp(0, v, 0x90, 0xF, 0xF, false);  // quad_perm [0,0,1,2]
    v += sub >= 1 ? o : 0;
    o = __builtin_amdgcn_update_dpp(0, v, 0x44, 0xF, 0xF, false);  // quad_perm [0,1,0,1]
    return v + (sub >= 2 ? o : 0);
}

// rows r = 3 xi + yi over the cells within one of the query's in the first
// (and second) index dimension, each a run of the last one's cells within one:
// lane `sub` of the query's quad takes rows sub, sub + 4 and 8; every row's two
// offsets are loaded before any is used, so the runs cost one memory round trip
__device__ __forceinline__ void build_runs(const GridArg &G, const int *__restrict__ off, const float *qy, int stride,
                                           int sub, float s_star, int *q) {
    const int C = G.C;
    const float ecs = ecell_width(C);
    const int c0 = ecell_of(qy[G.tI[0] * stride], ecs, C);
    const int c1 = G.j == 3 ? ecell_of(qy[G.tI[1] * stride], ecs, C) : 0;
    const float yl = qy[G.tI[G.j - 1] * stride];
    const int cl = ecell_of(yl, ecs, C);
    const int F = G.F > 1 ? G.F : 1, CF = C * F;
    // a run: the buckets of the last dimension's cells within one of the
    // query's, less those farther than eps from the query's coordinate (a
    // neighbour's squared difference there is at most s_star; the bounds are
    // rounded outwards and the bucket map is monotone, so no neighbour is lost)
    int lo = max(cl - 1, 0) * F, hi = min(cl + 1, C - 1) * F + F - 1;
    if (F > 1) {
        const double xq = (double) yl;
        const double em = sqrt((double) s_star) * 1.001 + 1e-6;
        lo = max(lo, fine_key(__double2float_rd(xq - em), C, F));
        hi = min(hi, fine_key(__double2float_ru(xq + em), C, F));
    }
    const int x0 = max(c0 - 1, 0), nx = G.j == 1 ? 1 : min(c0 + 1, C - 1) - x0 + 1;
    const int y0 = max(c1 - 1, 0), ny = G.j == 3 ? min(c1 + 1, C - 1) - y0 + 1 : 1;
    int a[3], e[3];
#pragma unroll
    for (int w = 0; w < 3; ++w) {
        // rows past the edge of the grid load a row inside it (no branch
        // around the loads) and are emptied below
        const int r = min(sub + 4 * w, 8);
        const int xi = min(r / 3, nx - 1), yi = min(r % 3, ny - 1);
        const int row = G.j == 1 ? 0 : G.j == 2 ? (x0 + xi) * CF : ((x0 + xi) * C + y0 + yi) * CF;
        a[w] = off[row + lo];
        e[w] = off[row + hi + 1];
    }
    int acc = 0, gacc = 0;
#pragma unroll
    for (int w = 0; w < 3; ++w) {
        const int r = sub + 4 * w;
        const int len = r < 9 && r / 3 < nx && r % 3 < ny ? max(e[w] - a[w], 0) : 0;
        const int s = acc + quad_scan(len, sub), g = gacc + quad_scan((len + 3) >> 2, sub);
        if (r < 9) {
            q[r] = a[w];
            q[10 + r] = s;
            q[21 + r] = g;
        }
        acc = __builtin_amdgcn_update_dpp(0, s, 0xFF, 0xF, 0xF, false);  // quad_perm [3,3,3,3]
        gacc = __builtin_amdgcn_update_dpp(0, g, 0xFF, 0xF, 0xF, false);
    }
    if (sub == 0) {
        q[9] = 0;
        q[19] = G.j == 1 ? 0 : 3 * (c0 - x0) + (G.j == 3 ? c1 - y0 : 0);
        q[20] = 0;
    }
}

__device__ __forceinline__ int run_pos(const int *q, int c, int &r) {
    while (c >= q[10 + r]) ++r;
    return q[r] + (c - q[9 + r]);
}

// Candidate at local sorted position jj against the staged query: the cells of
// the checked dimensions within one of the query's (its coordinate between two
// cell edges), then the distance summed in subspace order with separate
// multiplies and adds, compared with s_star.
__device__ __forceinline__ bool cand_test(const BatchSub &B, const float *qy, const float2 *qc, int stride, int jj, float s_star, float &acc_out) {
    const int k = B.S.k;
    float acc = 0.0f;
    for (int t = 0; t < k; ++t) {
        const float y = B.col[t][jj];
        const float2 c = qc[t * stride];
        if (!(y >= c.x && y < c.y)) return false;
        const float diff = qy[t * stride] - y;
        const float sq = diff * diff;
        acc = acc + sq;
        if (acc > s_star) return false;
    }
    acc_out = acc;
    return true;
}

// LDS of the neighbour passes: per query k cell intervals, k coordinates and
// its runs
__device__ __forceinline__ void lds_layout(char *smem, int k, float2 *&sc, float *&sy, int *&qr) {
    sc = reinterpret_cast<float2 *>(smem);
    sy = reinterpret_cast<float *>(smem + sizeof(float2) * QPB * (size_t) k);
    qr = reinterpret_cast<int *>(smem + (sizeof(float2) + sizeof(float)) * QPB * (size_t) k);
}

// The query at sorted position i into LDS, by its quad: the coordinates and,
// per checked dimension, the interval [lower, upper) of the coordinates whose
// eps cell is within one of its own (lane `sub` takes dimensions sub, sub + 4,
// ...; the cells come from the coordinates with the discretisation's formula,
// the intervals from the table of cell edges, see cell_edge), then its runs.
// By one lane of the four it took four times a wave's instructions: n=100,000
// d=20, the full link phase 34.1 -> 28.1 ms a run, the counts of k_b_count 45.7 ->
// 43.0; n=25,000 d=15 1.2 -> 1.1 and 1.2 -> 1.2.
__device__ __forceinline__ void stage_query_b(const BatchSub &B, const float *__restrict__ edge, int i, int sub,
                                              float s_star, float *sy, float2 *sc, int stride, int *q) {
    const int k = B.S.k;
    const float ecs = ecell_width(B.G.C);
    const float inf = __builtin_inff();
    for (int t0 = 0; t0 < k; t0 += 2 * kBLanes) {
        // two dimensions' loads are issued before any store (a store to LDS
        // through a generic pointer would order the second load after it)
        const int t1 = t0 + sub, t2 = t1 + kBLanes;
        const float y1 = t1 < k ? B.col[t1][i] : 0.0f, y2 = t2 < k ? B.col[t2][i] : 0.0f;
        float2 i1 = make_float2(-inf, inf), i2 = i1;
        if (t1 < k && ((B.G.checkmask >> t1) & 1ull)) {
            const int e = ecell_of(y1, ecs, B.G.C);
            i1 = make_float2(edge[e], edge[e + 3]);
        }
        if (t2 < k && ((B.G.checkmask >> t2) & 1ull)) {
            const int e = ecell_of(y2, ecs, B.G.C);
            i2 = make_float2(edge[e], edge[e + 3]);
        }
        if (t1 < k) {
            sy[t1 * stride] = y1;
            sc[t1 * stride] = i1;
        }
        if (t2 < k) {
            sy[t2 * stride] = y2;
            sc[t2 * stride] = i2;
        }
    }
    wave_sync();
    build_runs(B.G, B.off, sy, stride, sub, s_star, q);
    wave_sync();
}

// ------------------------------------------------------------ candidate walks of one query
// The LPQ lanes of a query take candidates c0 + u*LPQ + sub of each step.
// The walk starts at a pseudo-random candidate of the run of the query's own
// cells (the densest part of its neighbourhood) and wraps: the first
// neighbours found are then spread over the candidates (random sample edges
// for the components pass, as Afforest draws them) instead of the same few
// points at the start of a shared run.
struct QueryWalk {
    const BatchSub &B;
    int n, i, p;
    const int *q;    // the query's runs (LDS)
    const float *qy;   // its coordinates (LDS, stride QPB)
    const float2 *qc;  // its cell intervals (LDS, stride QPB)
    float s_star, eps;
    double phirel;
    int *nbp;        // its two recorded neighbours
};

__device__ __forceinline__ int walk_rot(const QueryWalk &W, int total) {
    const int *q = W.q;
    const int cs0 = q[9 + q[19]], clen = q[10 + q[19]] - cs0;
    return total > 0 ? cs0 + (int) (((uint32_t) W.p * 2654435761u) % (uint32_t) max(clen, 1)) : 0;
}

// neighbours found in one step: the first kSampleEdges are recorded (the sample edges
// of the components pass); phi adds the terms of the step
template <int U, bool PHI>
__device__ __forceinline__ void walk_tally(const QueryWalk &W, const int (&jj)[U], const bool (&hit)[U],
                                           const float (&accs)[U], int &found, double &dsum) {
    constexpr int LPQ = kBLanes;
    const int sub = __lane_id() % LPQ;
    const int gshift = (__lane_id() / LPQ) * LPQ;
    const unsigned long long below = (1ull << sub) - 1ull;
    if (PHI) {
        double part = 0.0;
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (hit[u]) part += phi_term(accs[u], W.eps);
        for (int o = LPQ / 2; o > 0; o >>= 1) part += __shfl_xor(part, o);
        dsum += part;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const unsigned long long mine = (__ballot(hit[u]) >> gshift) & ((1ull << LPQ) - 1ull);
        if (hit[u] && found < kSampleEdges) {
            const int at = found + __popcll(mine & below);
            if (at < kSampleEdges) W.nbp[at] = W.B.order[jj[u]];
        }
        found += __popcll(mine);
    }
}

__device__ __forceinline__ bool walk_more(const QueryWalk &W, bool phi, int found, double dsum, int total) {
    if (phi) {
        // phi may stop once its running double sum is certainly above both thresholds
        const double thr_max = (double) fmaxf(W.B.phi_w, W.B.phi_d);
        return dsum * (1.0 - (double) total * W.phirel) < thr_max;
    }
    return found < W.B.cap;
}

// The cell test of a step's hits.  A candidate within eps lies more than one
// cell away only next to a cell edge, so the test runs on the few candidates
// that passed the distance: its coordinates are read again there (they were
// just loaded) rather than kept in registers for all of them.
template <int U>
__device__ __forceinline__ void cells_of_hits(const BatchSub &B, const float2 *qc, int stride, uint32_t checked,
                                              int jj0, bool (&hit)[U]) {
    typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
    static_assert(U == 4, "one 16-byte load per column");
    if (!(hit[0] | hit[1] | hit[2] | hit[3])) return;
    for (uint32_t m = checked; m; m &= m - 1) {
        const int t = __builtin_ctz(m);
        const float2 c = qc[t * stride];
        const f4u y = *reinterpret_cast<const f4u *>(B.col[t] + (uint32_t) jj0);
#pragma unroll
        for (int u = 0; u < U; ++u) hit[u] = hit[u] & (y[u] >= c.x) & (y[u] < c.y);
    }
}

// k = K dimensions (the host checks), counts or phi.  Each lane takes four
// consecutive candidates of one run per step, so a step loads each coordinate
// column with one 16-byte load per lane instead of four 4-byte loads, and
// nothing else: the eps cells of the checked dimensions are tested on the
// coordinates of the step's hits (cells_of_hits).
// Load instructions are what these walks pay for most (the CUs' address unit is busy
// for 63 to 79% of the cycles, at 24 to 29 cycles and 12 to 21 cache lines a load;
// n=100,000 d=20).  The runs are
// concatenated in groups of four (q[20..29]); the last group of a run masks
// the positions past the run's end, which are read (up to three past the
// run: the batch's coordinate buffer ends with padding) but
// never counted.  A lane's first group position is 4-byte aligned only;
// dword-aligned multi-dword global loads are supported on gfx950.
template <int K, bool PHI>
__device__ __forceinline__ void walk_vec(const QueryWalk &W, int &found, double &dsum, bool &more, long long &seen) {
    typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
    constexpr int LPQ = kBLanes, U = 4;
    const BatchSub &B = W.B;
    const uint32_t checked = (uint32_t) B.G.checkmask;
    const int *q = W.q;
    const int sub = __lane_id() % LPQ;
    const int gtotal = q[29], total = q[18];
    // start at a pseudo-random group of the query's own run (spreads the
    // sample edges), walk to the end, then from the start to there
    const int own = q[19];
    const int og = q[20 + own], olen = q[21 + own] - og;
    const int grot = gtotal > 0 ? og + (int) (((uint32_t) W.p * 2654435761u) % (uint32_t) max(olen, 1)) : 0;
    const float *col[K];
    float qv[K];
#pragma unroll
    for (int t = 0; t < K; ++t) {
        col[t] = B.col[t];
        qv[t] = W.qy[t * QPB];
    }
    for (int segm = 0; segm < 2; ++segm) {
        const int gbeg = segm == 0 ? grot : 0, gend = segm == 0 ? gtotal : grot;
        int r = segm == 0 ? own : 0;
        int rgend = q[21 + r];
        for (int g0 = gbeg; g0 < gend && more; g0 += LPQ) {
            const int g = min(g0 + sub, gend - 1);
            while (g >= rgend) {
                ++r;
                rgend = q[21 + r];
            }
            const int e0 = (g - q[20 + r]) << 2;  // the group's first element in run r
            const int len = q[10 + r] - q[9 + r];
            const int nv = g0 + sub < gend ? min(U, len - e0) : 0;  // its elements inside the run
            const int jj0 = q[r] + e0;
            f4u y[K];
#pragma unroll
            for (int t = 0; t < K; ++t)
                y[t] = *reinterpret_cast<const f4u *>(reinterpret_cast<const char *>(col[t]) +
                                                      ((uint32_t) jj0 << 2));
            int jj[U];
            bool hit[U];
            float accs[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                float acc = 0.0f;
#pragma unroll
                for (int t = 0; t < K; ++t) {
                    const float diff = qv[t] - y[t][u];
                    const float sq = diff * diff;
                    acc = acc + sq;
                }
                jj[u] = jj0 + u;
                hit[u] = (u < nv) & (jj[u] != W.i) & (acc <= W.s_star);
                accs[u] = acc;
            }
            if (checked) cells_of_hits<U>(B, W.qc, QPB, checked, jj0, hit);
            // the query's examined candidates of the step, summed over its
            // quad with two DPP moves
            int ex = nv;
            ex += __builtin_amdgcn_update_dpp(0, ex, 0xB1, 0xF, 0xF, false);  // quad_perm [1,0,3,2]
            ex += __builtin_amdgcn_update_dpp(0, ex, 0x4E, 0xF, 0xF, false);  // quad_perm [2,3,0,1]
            // the query's hits, summed over the quad with two DPP moves (phi:
            // and the step's phi terms); the ballots of walk_tally only while
            // the two sample edges are open
            int h = 0;
#pragma unroll
            for (int u = 0; u < U; ++u) h += hit[u] ? 1 : 0;
            h += __builtin_amdgcn_update_dpp(0, h, 0xB1, 0xF, 0xF, false);
            h += __builtin_amdgcn_update_dpp(0, h, 0x4E, 0xF, 0xF, false);
            if (PHI) {
                double part = 0.0;
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (hit[u]) part += phi_term(accs[u], W.eps);
                part += __shfl_xor(part, 1);
                part += __shfl_xor(part, 2);
                dsum += part;
            }
            if (found < kSampleEdges && h > 0) {
                double unused = 0.0;
                int f = found;
                walk_tally<U, false>(W, jj, hit, accs, f, unused);
            }
            found += h;
            seen += ex;
            more = walk_more(W, PHI, found, dsum, total);
        }
    }
}

// any k, one candidate per lane at a time (cand_test)
template <bool PHI>
__device__ __forceinline__ void walk_generic(const QueryWalk &W, int &found, double &dsum, bool &more,
                                             long long &seen) {
    constexpr int LPQ = kBLanes, U = 4, STEP = LPQ * U;
    const int *q = W.q;
    const int sub = __lane_id() % LPQ;
    const int total = q[18];
    const int rot = walk_rot(W, total);
    int r = 0;
    bool wrapped = false;
    for (int c0 = 0; c0 < total && more; c0 += STEP) {
        int jj[U];
        bool hit[U];
        float accs[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = c0 + u * LPQ + sub;
            jj[u] = -1;
            if (c < total) {
                int cr = c + rot;
                if (cr >= total) {
                    cr -= total;
                    if (!wrapped) {
                        wrapped = true;
                        r = 0;
                    }
                }
                jj[u] = run_pos(q, cr, r);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            accs[u] = 0.0f;
            hit[u] = jj[u] >= 0 && jj[u] != W.i &&
                     cand_test(W.B, W.qy, W.qc, QPB, jj[u], W.s_star, accs[u]);
        }
        walk_tally<U, PHI>(W, jj, hit, accs, found, dsum);
        seen += min(STEP, total - c0);
        more = walk_more(W, PHI, found, dsum, total);
    }
}

// ------------------------------------------------------------ neighbour counts
// LIST = the compacted queries of each subspace (blocks by segment), else every
// sorted position of subspace blockIdx.y whose count is still missing
// (components pass, with the subset bound).
template <bool LIST, bool PHI, int K>
__global__ __launch_bounds__(kBlock) void k_b_count(const BatchSub *__restrict__ subs, const int *__restrict__ blk_off,
                                                    int nsub, int n, const float *__restrict__ edge,
                                                    const int *__restrict__ qlist, const int *__restrict__ qstart,
                                                    float s_star, float eps, double phirel, int *__restrict__ nb,
                                                    int2 *__restrict__ fb, int *__restrict__ nfb, int fbcap,
                                                    unsigned long long *__restrict__ stat) {
    constexpr int LPQ = kBLanes;
    extern __shared__ char smem[];
    int b, blk;
    if (LIST) {
        b = seg_of(blk_off, nsub, blockIdx.x);
        blk = blockIdx.x - blk_off[b];
    } else {
        b = blockIdx.y;
        blk = blockIdx.x;
    }
    const BatchSub &B = subs[b];
    const int k = B.S.k;
    float2 *sc;
    float *sy;
    int *qr;
    lds_layout(smem, k, sc, sy, qr);
    const int lq = threadIdx.x / LPQ, sub = threadIdx.x % LPQ;
    int i = 0;
    bool active;
    if (LIST) {
        const int q = qstart[b] + blk * QPB + lq;
        active = q < qstart[b + 1];
        if (active) i = (int) (qlist[q] - B.base);
    } else {
        i = blk * QPB + lq;
        active = i < n;
    }
    int *cnt = B.cnt;
    const int p = active ? B.order[i] : 0;
    active = active && cnt[p] < 0;
    // N_S(p) is a subset of N_S'(p) for S' a subset of S: the smallest
    // complete count of the subspaces S minus one dimension, when below both
    // thresholds of S, decides p without a scan (and stays an upper bound);
    // phi: the smallest stored upper bound, below both phi thresholds
    if (active && B.nbound > 0) {
        int bb = INT_MAX;
        for (int t = 0; t < B.nbound; ++t) {
            const int v = B.bound[t][p];
            if (v >= 0) bb = min(bb, PHI ? v >> 2 : v);
        }
        if (PHI ? bb < kPhiNoBound && (double) bb * 0.25 < (double) fminf(B.phi_w, B.phi_d) : bb < B.lo) {
            if (sub == 0) cnt[p] = PHI ? bb << 2 : bb;
            active = false;
        }
    }
    int *q = qr + lq * kRangeWords;
    if (active) stage_query_b(B, edge, i, sub, s_star, sy + lq, sc + lq, QPB, q);
    long long seen = 0;
    int found = 0;
    if (active) {
        double dsum = 0.0;
        bool more = true;
        const QueryWalk W{B, n, i, p, q, sy + lq, sc + lq, s_star, eps, phirel,
                          nb + kSampleEdges * (B.nbase + p)};
        // K > 0: every subspace of the launch has k = K (the host checks), so
        // the walk is compiled for it
        if constexpr (K > 0)
            walk_vec<K, PHI>(W, found, dsum, more, seen);
        else
            walk_generic<PHI>(W, found, dsum, more, seen);
        if (PHI) {
            // decision bits: 1 weak-dense, 2 dense; a threshold inside the
            // rounding band sends the point to the leaf-order recomputation
            const double lo = dsum * (1.0 - (double) found * phirel);
            const double hi = dsum * (1.0 + (double) found * phirel);
            int code = 0;
            bool unsure = false;
            double ub = -1.0;  // stopped early: no bound
            if (!more) {
                code = 3;
            } else {
                const double tw = (double) B.phi_w, td = (double) B.phi_d;
                if (lo >= tw) code |= 1;
                else if (!(hi < tw)) unsure = true;
                if (lo >= td) code |= 2;
                else if (!(hi < td)) unsure = true;
                // hi bounds T, the exact sum of the terms (the double scan-order
                // sum is within N 2^-52 of it)
                ub = hi * (1.0 + (double) found * phirel);
            }
            if (sub == 0) {
                cnt[p] = phi_code(code, ub);
                if (unsure) {
                    const int at = atomicAdd(nfb, 1);
                    if (at < fbcap) fb[at] = make_int2(b, p);
                }
            }
        } else if (sub == 0) {
            cnt[p] = found;
        }
    }
    if (stat) {
        // per wave into one of 64 slot groups: [0] candidates examined, [1]
        // points counted, [2] algorithmic bytes (4k + 4 per point, 4 + 4k per
        // neighbour established), [3] bytes of the examined candidates (k coordinates)
        const bool mine = sub == 0 && active;
        long long done = mine ? 1 : 0;
        long long abytes = mine ? (4ll * k + 4) + (long long) found * (4 + 4ll * k) : 0;
        if (sub != 0) seen = 0;
        long long ebytes = seen * 4ll * k;
        for (int o = 32; o > 0; o >>= 1) {
            seen += __shfl_down(seen, o);
            done += __shfl_down(done, o);
            abytes += __shfl_down(abytes, o);
            ebytes += __shfl_down(ebytes, o);
        }
        if (__lane_id() == 0 && done) {
            unsigned long long *slot = stat + 16 * (blockIdx.x & 63);
            atomicAdd(&slot[0], (unsigned long long) seen);
            atomicAdd(&slot[1], (unsigned long long) done);
            atomicAdd(&slot[2], (unsigned long long) abytes);
            atomicAdd(&slot[3], (unsigned long long) ebytes);
        }
    }
}

// ------------------------------------------------------------ neighbour counts of all children of a mask
// The children S | {m} of a frontier mask S count the same points (those of
// S's trees), and a neighbour in S | {m} is a neighbour in S whose coordinate
// in m is near too; m is above every dimension of S, so the distance of the
// child is S's running sum plus one last term.  One walk over the candidates of
// S therefore serves all children: the kFanLanes lanes of a query test
// kFanLanes * 4 candidates of S per step (the grouped loads of walk_vec) and
// put the few neighbours found into LDS; then every lane, standing for NC
// children and one of kFanLanes / CW slots, adds m's term of the slot's
// neighbours: the lanes read consecutive coordinates of a neighbour's row of X.
// The walk ends when every child is decided (cap, phi) or the runs are done.
// A pair that the learned pruner skips is no child of its tree's points: they
// are not counted in it, and points without a live child make no walk.
// The children's bounds (k_b_count) are not looked up: one undecided child
// makes the walk anyway, and the look-up costs a scattered read per child and
// bound (n=100,000 d=20, masks of three dimensions: 54 ms with it, 49 without).
// Bound: no unit alone (n=100,000 d=20 eps=0.02): waves wait for 60 to 68% of
// their cycles (a query's set-up is a chain of dependent loads), while the CUs'
// address units are busy for 73 to 81% (18 cycles and 8 to 14 cache lines a load)
// and VALU instructions issue at 0.67 to 0.81 of one a SIMD per four cycles.
// Masks of few children have slots instead of idle lanes (49 -> 43 ms; by
// child, k_b_count took 63 ms).
// Six waves a SIMD in count mode with up to two children a lane, up to K = 6:
// 91 -> 79 VGPRs at K = 2, eight children.  The 80 registers of six waves are enough
// or two short up to K = 4; at K = 5 up to 10 are spilled, at K = 6 8 to 17.  Whole
// runs at n=100,000 d=20 eps=0.02: without it 583 ms, up to K = 4 583 and 578, K = 5
// 575 and 574, K = 6 576 and 575 (the last neither gains nor costs); n=25,000 d=15
// 9.96 -> 9.80 ms of kernels; seven waves 591, eight 623, and four children a lane
// spill 21 registers or more at six.
template <bool PHI, int K, int CW, int NC>
__global__ __launch_bounds__(kBlock, PHI || NC > 2 || K > 6 ? 3 : 6) void k_b_fan(const BatchSub *__restrict__ groups, const FanJob *__restrict__ jobs,
                                                  const int *__restrict__ blk_off, int njob, FanTable T, int d,
                                                  const float *__restrict__ X, const float *__restrict__ edge,
                                                  const int *__restrict__ qlist, const int *__restrict__ qstart,
                                                  float s_star, float eps, double phirel, int cap, float phi_w,
                                                  float phi_d, int *__restrict__ nb, int2 *__restrict__ fb,
                                                  int *__restrict__ nfb, int fbcap,
                                                  unsigned long long *__restrict__ stat) {
    typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
    typedef int i4u __attribute__((ext_vector_type(4), aligned(4)));
    constexpr int L = kFanLanes, Q = kFanQueries, U = 4;
    constexpr int HS = L / CW;  // slots: neighbours of the step taken at once
    __shared__ float sy[K][Q];
    __shared__ float2 sc[K][Q];
    __shared__ int rs[9][Q], rl[9][Q], rg[10][Q];  // runs: first position, length, groups of four before (rg[9]: all)
    __shared__ uint2 hits[Q][L * U + U * HS];      // (row offset in X, sum over S) of the step's neighbours in S
    const int ji = seg_of(blk_off, njob, blockIdx.x);
    const FanJob J = jobs[ji];
    const BatchSub &B = groups[J.g];
    const int lq = threadIdx.x / L, l = threadIdx.x % L;
    const int slot = l / CW, cl = l % CW;
    const int gshift = __lane_id() & ~(L - 1);
    const int qi = qstart[J.g] + (blockIdx.x - blk_off[ji]) * Q + lq;
    bool active = qi < qstart[J.g + 1];
    int seen = 0, nhits = 0;
    // a lane without a live child in place c starts its count at kNone, more than
    // any count and its sum over the slots in range (n <= kFanPoints; the host
    // checks): the walk does not wait for it and records no edges
    constexpr int kNone = kFanPoints;
    static_assert((long long) kNone * (HS + 1) < INT_MAX, "the slots' counts are summed");
    int found[NC];
    const int at = active ? qlist[qi] : 0;
    {
        unsigned long long live = J.nch < 64 ? (1ull << J.nch) - 1ull : ~0ull;
        if (T.live && active) live &= T.live[2 * T.seg[at] + J.part];
        active = active && live != 0;
#pragma unroll
        for (int c = 0; c < NC; ++c) found[c] = (live >> (cl + CW * c)) & 1ull ? 0 : kNone;
    }
    if (active) {
        const int i = (int) (at - B.base);
        const int p = B.order[i];
        // the query's coordinates and cell intervals in S: lane t holds dimension t
        const float inf = __builtin_inff();
        const float ecs = ecell_width(B.G.C);
        if (l < K) {
            const float y = B.col[l][i];
            float2 c = make_float2(-inf, inf);
            if ((B.G.checkmask >> l) & 1ull) {
                const int e = ecell_of(y, ecs, B.G.C);
                c = make_float2(edge[e], edge[e + 3]);
            }
            sy[l][lq] = y;
            sc[l][lq] = c;
        }
        // the lane's children: the query's coordinate in m and the interval of
        // the cells around its own
        int ch[NC], dim[NC];
        float xq[NC], lo[NC], hi[NC];
        double dsum[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            ch[c] = J.ch0 + min(cl + CW * c, J.nch - 1);
            dim[c] = T.dim[ch[c]];
            xq[c] = X[(size_t) p * d + dim[c]];
            const int e = ecell_of(xq[c], ecs, B.G.C);
            lo[c] = edge[e];
            hi[c] = edge[e + 3];
            dsum[c] = 0.0;
        }
        wave_sync();
        // the runs of build_runs, lane r (of nine) row r
        int gtotal, own, ogrp, olen, total;
        {
            const GridArg &G = B.G;
            const int C = G.C;
            const int c0 = ecell_of(sy[G.tI[0]][lq], ecs, C);
            const int c1 = G.j == 3 ? ecell_of(sy[G.tI[1]][lq], ecs, C) : 0;
            const float yl = sy[G.tI[G.j - 1]][lq];
            const int cc = ecell_of(yl, ecs, C);
            const int F = G.F > 1 ? G.F : 1, CF = C * F;
            int clo = max(cc - 1, 0) * F, chi = min(cc + 1, C - 1) * F + F - 1;
            if (F > 1) {
                const double em = sqrt((double) s_star) * 1.001 + 1e-6;
                clo = max(clo, fine_key(__double2float_rd((double) yl - em), C, F));
                chi = min(chi, fine_key(__double2float_ru((double) yl + em), C, F));
            }
            const int x0 = max(c0 - 1, 0), nx = G.j == 1 ? 1 : min(c0 + 1, C - 1) - x0 + 1;
            const int y0 = max(c1 - 1, 0), ny = G.j == 3 ? min(c1 + 1, C - 1) - y0 + 1 : 1;
            own = G.j == 1 ? 0 : 3 * (c0 - x0) + (G.j == 3 ? c1 - y0 : 0);
            const int xi = l / 3, yi = l % 3;
            int a = 0, len = 0;
            if (xi < nx && yi < ny) {
                const int row = G.j == 1 ? 0 : G.j == 2 ? (x0 + xi) * CF : ((x0 + xi) * C + y0 + yi) * CF;
                a = B.off[row + clo];
                len = max(B.off[row + chi + 1] - a, 0);
            }
            const int g = (len + U - 1) / U;
            int incl = g;
            total = len;
            for (int o = 1; o < L; o <<= 1) {
                const int v = __shfl_up(incl, o, L);
                if (l >= o) incl += v;
                total += __shfl_xor(total, o, L);
            }
            if (l < 9) {
                rs[l][lq] = a;
                rl[l][lq] = len;
                rg[l][lq] = incl - g;
            }
            if (l == 9) rg[9][lq] = incl;
            gtotal = __shfl(incl, 9, L);
            ogrp = __shfl(incl - g, own, L);
            olen = __shfl(g, own, L);
        }
        wave_sync();
        const float *col[K];
        float qv[K];
#pragma unroll
        for (int t = 0; t < K; ++t) {
            col[t] = B.col[t];
            qv[t] = sy[t][lq];
        }
        const uint32_t checked = (uint32_t) B.G.checkmask;
        const unsigned long long below = (1ull << l) - 1ull;
        const uint2 none = make_uint2((uint32_t) p * (uint32_t) d, __float_as_uint(inf));
        // start at a pseudo-random group of the query's own run (spreads the
        // sample edges), walk to the end, then from the start to there
        const int grot = gtotal > 0 ? ogrp + (int) (((uint32_t) p * 2654435761u) % (uint32_t) max(olen, 1)) : 0;
        bool more = true;
        for (int segm = 0; segm < 2; ++segm) {
            const int gbeg = segm == 0 ? grot : 0, gend = segm == 0 ? gtotal : grot;
            int r = segm == 0 ? own : 0;
            for (int g0 = gbeg; g0 < gend && more; g0 += L) {
                const int g = min(g0 + l, gend - 1);
                while (g >= rg[r + 1][lq]) ++r;
                const int e0 = (g - rg[r][lq]) * U;
                const int nv = g0 + l < gend ? min(U, rl[r][lq] - e0) : 0;
                const int jj0 = rs[r][lq] + e0;
                f4u y[K];
#pragma unroll
                for (int t = 0; t < K; ++t) y[t] = *reinterpret_cast<const f4u *>(col[t] + (uint32_t) jj0);
                bool hit[U];
                float accs[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    float acc = 0.0f;
#pragma unroll
                    for (int t = 0; t < K; ++t) {
                        const float diff = qv[t] - y[t][u];
                        const float sq = diff * diff;
                        acc = acc + sq;
                    }
                    hit[u] = (u < nv) & (jj0 + u != i) & (acc <= s_star);
                    accs[u] = acc;
                }
                if (checked) cells_of_hits<U>(B, &sc[0][lq], Q, checked, jj0, hit);
                seen += nv;
                i4u id = {0, 0, 0, 0};
                if (hit[0] | hit[1] | hit[2] | hit[3])
                    id = *reinterpret_cast<const i4u *>(B.order + (uint32_t) jj0);
                int nh = 0;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const unsigned long long m = (__ballot(hit[u]) >> gshift) & 0xFFFFull;
                    if (hit[u])
                        hits[lq][nh + __popcll(m & below)] =
                            make_uint2((uint32_t) id[u] * (uint32_t) d, __float_as_uint(accs[u]));
                    nh += __popcll(m);
                }
                if (nh == 0) continue;  // uniform over the query's lanes
                if (l < U * HS) hits[lq][nh + l] = none;  // past the last one: never near
                wave_sync();
                nhits += nh;
                for (int h0 = 0; h0 < nh; h0 += U * HS) {
                    uint2 e[U];
                    float z[U][NC];
#pragma unroll
                    for (int u = 0; u < U; ++u) e[u] = hits[lq][h0 + u * HS + slot];
#pragma unroll
                    for (int u = 0; u < U; ++u)
#pragma unroll
                        for (int c = 0; c < NC; ++c) z[u][c] = X[e[u].x + (uint32_t) dim[c]];
#pragma unroll
                    for (int u = 0; u < U; ++u)
#pragma unroll
                        for (int c = 0; c < NC; ++c) {
                            const float diff = xq[c] - z[u][c];
                            const float sq = diff * diff;
                            const float acc = __uint_as_float(e[u].y) + sq;
                            if (acc <= s_star && z[u][c] >= lo[c] && z[u][c] < hi[c]) {
                                // sample edges: the first of slots 0 and 1, or the first two of the only slot
                                if (HS > 1 ? (slot < kSampleEdges && found[c] == 0) : found[c] < kSampleEdges)
                                    nb[kSampleEdges * (T.nbase[ch[c]] + p) + (HS > 1 ? slot : found[c])] =
                                        (int) (e[u].x / (uint32_t) d);
                                ++found[c];
                                if (PHI) dsum[c] += phi_term(acc, eps);
                            }
                        }
                }
                // undecided children, over the slots
                bool open = false;
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    if (PHI) {
                        double ds = dsum[c];
                        for (int o = CW; o < L; o <<= 1) ds += __shfl_xor(ds, o);
                        open |= (found[c] < kNone) &
                                (ds * (1.0 - (double) total * phirel) < (double) fmaxf(phi_w, phi_d));
                    } else {
                        int f = found[c];
                        for (int o = CW; o < L; o <<= 1) f += __shfl_xor(f, o);
                        open |= f < cap;
                    }
                }
                more = ((__ballot(open) >> gshift) & 0xFFFFull) != 0;
                wave_sync();
            }
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            for (int o = CW; o < L; o <<= 1) found[c] += __shfl_xor(found[c], o);
            if (PHI)
                for (int o = CW; o < L; o <<= 1) dsum[c] += __shfl_xor(dsum[c], o);
            if (slot != 0 || found[c] >= kNone) {
                found[c] = -1;  // counted by another lane, or a skipped pair
                continue;
            }
            if (PHI) {
                // as in k_b_count; a sum above both thresholds may be incomplete
                const double tw = (double) phi_w, td = (double) phi_d;
                const double sl = dsum[c] * (1.0 - (double) found[c] * phirel);
                const double sh = dsum[c] * (1.0 + (double) found[c] * phirel);
                int code = 0;
                bool unsure = false;
                double ub = -1.0;
                if (!(dsum[c] * (1.0 - (double) total * phirel) < (double) fmaxf(phi_w, phi_d))) {
                    code = 3;
                } else {
                    if (sl >= tw) code |= 1;
                    else if (!(sh < tw)) unsure = true;
                    if (sl >= td) code |= 2;
                    else if (!(sh < td)) unsure = true;
                    ub = sh * (1.0 + (double) found[c] * phirel);
                }
                T.cnt[ch[c]][p] = phi_code(code, ub);
                if (unsure) {
                    const int at = atomicAdd(nfb, 1);
                    if (at < fbcap) fb[at] = make_int2(ch[c], p);
                }
            } else {
                T.cnt[ch[c]][p] = found[c];
            }
        }
    }
    if (stat) {
        // the slots of k_b_count: candidates of S examined, (child, point)
        // pairs counted, their algorithmic bytes, bytes of the examined
        // candidates (their K coordinates; a neighbour's id and its
        // coordinates in the children's dimensions)
        long long done = 0, abytes = 0;
#pragma unroll
        for (int c = 0; c < NC; ++c)
            if (active && found[c] >= 0) {
                done += 1;
                abytes += (4ll * (K + 1) + 4) + (long long) found[c] * (4 + 4ll * (K + 1));
            }
        long long sn = seen;
        long long ebytes = sn * 4ll * K + (l == 0 ? (long long) nhits * (4 + 4ll * J.nch) : 0);
        for (int o = 32; o > 0; o >>= 1) {
            sn += __shfl_down(sn, o);
            done += __shfl_down(done, o);
            abytes += __shfl_down(abytes, o);
            ebytes += __shfl_down(ebytes, o);
        }
        if (__lane_id() == 0 && done) {
            unsigned long long *slot_at = stat + 16 * (blockIdx.x & 63);
            atomicAdd(&slot_at[0], (unsigned long long) sn);
            atomicAdd(&slot_at[1], (unsigned long long) done);
            atomicAdd(&slot_at[2], (unsigned long long) abytes);
            atomicAdd(&slot_at[3], (unsigned long long) ebytes);
        }
    }
}

// ------------------------------------------------------------ dense components of a batch
// (grid.y = subspace)

// The sample phase of one subspace (the unions of the sample edges, compressed
// parents, the giant component) in one block, with the union-find in LDS: a
// device-scope swap goes past the XCD's L2 and their rate bounded the same
// unions on global parents (n=100,000 d=20, 29 batches: 41.5 ms there).  One
// block's loads in flight bound it, so every pass takes kUfItems points a thread
// (one 32.0 ms, four 28.4), and what needs no LDS runs on the whole chip: above
// kUfCap points every point first takes the smallest of itself and its dense
// sample neighbours as parent (k_b_dense_init; each thread writes its own entry,
// a forest without a swap, about a third of the points are left as roots), and
// the block numbers the roots in id order for the LDS (smaller number = smaller
// id, so roots stay the smallest ids): 13.3 ms and 10.6 around it.  A subspace
// with more roots than fit clears fit[s] and is left to the global passes.
constexpr int kUfCap = 39936;
constexpr int kUfThreads = 1024, kUfWaves = kUfThreads / 64, kUfItems = 4;
__device__ __forceinline__ int lds_find(volatile int *up, int x) {
    int p = up[x];
    while (p != x) {
        const int g = up[p];
        if (g != p) up[x] = g;
        x = p;
        p = g;
    }
    return x;
}
__device__ __forceinline__ void lds_union(int *up, int a, int b) {
    while (true) {
        a = lds_find(up, a);
        b = lds_find(up, b);
        if (a == b) return;
        if (a > b) {
            const int t = a;
            a = b;
            b = t;
        }
        const int old = atomicCAS(&up[b], b, a);
        if (old == b) return;
        b = old;
    }
}
// point i's first parent: the smallest of itself and its dense sample neighbours
// (-1 when it is not dense)
__device__ __forceinline__ int hooked(const BatchSub &B, const int *__restrict__ nb, int i) {
    if (!meets(B.cnt[i], B.thr_dense, B.dbit)) return -1;
    int root = i;
#pragma unroll
    for (int e = 0; e < kSampleEdges; ++e) {
        const int q = nb[kSampleEdges * (B.nbase + i) + e];
        if (q >= 0 && q < root && meets(B.cnt[q], B.thr_dense, B.dbit)) root = q;
    }
    return root;
}

__global__ __launch_bounds__(kUfThreads) void k_b_sample(const BatchSub *__restrict__ subs, int n,
                                                         const int *__restrict__ nb, int *__restrict__ rootpos,
                                                         int *__restrict__ par, int *__restrict__ giant,
                                                         int *__restrict__ fit) {
    __shared__ int up[kUfCap];
    __shared__ int wcnt[kUfWaves + 1];
    const BatchSub &B = subs[blockIdx.x];
    const int t = threadIdx.x, lane = __lane_id(), wv = t >> 6;
    int *pr = par + B.base;
    const bool numbered = n > kUfCap;  // uniform over the launch
    // every pass takes kUfItems points per thread at once: one block holds the
    // whole subspace, so its loads in flight bound it
    constexpr int M = kUfItems, STEP = kUfThreads * M;
    const int2 *nb2 = reinterpret_cast<const int2 *>(nb) + B.nbase;
    static_assert(kSampleEdges == 2, "a point's sample edges are one int2");
    if (!numbered) {
        for (int i0 = t; i0 < n; i0 += STEP) {
            int c[M];
#pragma unroll
            for (int u = 0; u < M; ++u) c[u] = B.cnt[min(i0 + u * kUfThreads, n - 1)];
#pragma unroll
            for (int u = 0; u < M; ++u) {
                const int i = i0 + u * kUfThreads;
                if (i >= n) continue;
                const bool dense = meets(c[u], B.thr_dense, B.dbit);
                pr[i] = dense ? i : -1;
                up[i] = i;
            }
        }
    } else {
        // roots of the wave's share (a multiple of 64), then their numbers:
        // csize[root] = number, comp[number] = root
        const int share = ((n + kUfWaves - 1) / kUfWaves + 63) & ~63;
        const int w0 = min(n, wv * share), w1 = min(n, w0 + share);
        int c = 0;
        for (int i = w0 + lane; i - lane < w1; i += 64) c += __popcll(__ballot(i < w1 && pr[i] == i));
        if (lane == 0) wcnt[wv] = c;
        __syncthreads();
        if (t == 0) {
            int acc = 0;
            for (int w = 0; w < kUfWaves; ++w) {
                const int v = wcnt[w];
                wcnt[w] = acc;
                acc += v;
            }
            wcnt[kUfWaves] = acc;
            fit[blockIdx.x] = acc <= kUfCap;
        }
        __syncthreads();
        if (wcnt[kUfWaves] > kUfCap) return;
        int at = wcnt[wv];
        for (int i = w0 + lane; i - lane < w1; i += 64) {
            const bool root = i < w1 && pr[i] == i;
            const unsigned long long m = __ballot(root);
            const int num = at + __popcll(m & ((1ull << lane) - 1ull));
            at += __popcll(m);
            if (root) {
                up[num] = num;
                B.csize[i] = num;
                B.comp[num] = i;
            }
        }
        __syncthreads();
        for (int i0 = t; i0 < n; i0 += STEP) {
            int r[M];
#pragma unroll
            for (int u = 0; u < M; ++u) r[u] = i0 + u * kUfThreads < n ? pr[i0 + u * kUfThreads] : -1;
#pragma unroll
            for (int u = 0; u < M; ++u)
                if (r[u] >= 0) r[u] = B.csize[r[u]];
#pragma unroll
            for (int u = 0; u < M; ++u)
                if (r[u] >= 0) pr[i0 + u * kUfThreads] = r[u];
        }
    }
    __syncthreads();
    for (int i0 = t; i0 < n; i0 += STEP) {
        int a[M], b[M][2];
        int2 q[M];
#pragma unroll
        for (int u = 0; u < M; ++u) {
            const int i = i0 + u * kUfThreads;
            a[u] = i < n ? pr[i] : -1;
            q[u] = i < n ? nb2[i] : make_int2(-1, -1);
        }
#pragma unroll
        for (int u = 0; u < M; ++u) {
            b[u][0] = a[u] >= 0 && q[u].x >= 0 && q[u].x < n ? pr[q[u].x] : -1;
            b[u][1] = a[u] >= 0 && q[u].y >= 0 && q[u].y < n ? pr[q[u].y] : -1;
        }
#pragma unroll
        for (int u = 0; u < M; ++u)
#pragma unroll
            for (int e = 0; e < 2; ++e)
                if (b[u][e] >= 0 && b[u][e] != a[u]) lds_union(up, a[u], b[u][e]);
    }
    __syncthreads();
    for (int i0 = t; i0 < n; i0 += STEP) {
        int r[M];
#pragma unroll
        for (int u = 0; u < M; ++u) r[u] = i0 + u * kUfThreads < n ? pr[i0 + u * kUfThreads] : -1;
#pragma unroll
        for (int u = 0; u < M; ++u)
            if (r[u] >= 0) r[u] = lds_find(up, r[u]);
        if (numbered) {
#pragma unroll
            for (int u = 0; u < M; ++u)
                if (r[u] >= 0) r[u] = B.comp[r[u]];
        }
#pragma unroll
        for (int u = 0; u < M; ++u)
            if (r[u] >= 0) pr[i0 + u * kUfThreads] = r[u];
    }
    __syncthreads();  // the ids by number are read, the parents written
    for (int i0 = t; !numbered && i0 < n; i0 += STEP) {
        int o[M];
#pragma unroll
        for (int u = 0; u < M; ++u) o[u] = B.order[min(i0 + u * kUfThreads, n - 1)];
#pragma unroll
        for (int u = 0; u < M; ++u) o[u] = pr[o[u]];
#pragma unroll
        for (int u = 0; u < M; ++u) {
            const int i = i0 + u * kUfThreads;
            if (i >= n) continue;
            rootpos[B.base + i] = o[u];
            B.csize[i] = 0;
        }
    }
    if (t < 256) {
        const int p = (int) (((long long) t * n) / 256);
        up[t] = p < n ? pr[p] : -1;
    }
    __syncthreads();
    if (t < 64) {
        // the most frequent of the 256 roots, the smaller id on a tie (k_b_giant)
        int bc = 0, br = -1;
        for (int u = t; u < 256; u += 64) {
            const int r = up[u];
            int c = 0;
            if (r >= 0)
                for (int v = 0; v < 256; ++v) c += up[v] == r;
            if (c > bc || (c == bc && c > 0 && r < br)) {
                bc = c;
                br = r;
            }
        }
        for (int o = 32; o > 0; o >>= 1) {
            const int c2 = __shfl_down(bc, o), r2 = __shfl_down(br, o);
            if (c2 > bc || (c2 == bc && c2 > 0 && r2 < br)) {
                bc = c2;
                br = r2;
            }
        }
        if (t == 0) giant[blockIdx.x] = bc > 0 ? br : -1;
    }
}

// First parents (hooked) of tables above kUfCap points.
__global__ void k_b_dense_init(const BatchSub *__restrict__ subs, int n, const int *__restrict__ nb,
                               int *__restrict__ par) {
    const BatchSub &B = subs[blockIdx.y];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) par[B.base + i] = hooked(B, nb, i);
}

// The sample edges on global parents, for the subspaces whose first parents do
// not fit (fit null: all).
// Sample phase of the components: every dense point links to the dense ones
// among the first kSampleEdges neighbours its count pass recorded (any edges would do:
// the full phase below links every point outside the giant component to all
// its dense neighbours, so the result does not depend on the sample).  It runs
// on compressed parents, so most edges are decided by two equal parents.
__global__ void k_b_link_sample(const BatchSub *__restrict__ subs, int n, const int *__restrict__ nb,
                                const int *__restrict__ fit, int *__restrict__ par) {
    if (fit && fit[blockIdx.y]) return;
    const BatchSub &B = subs[blockIdx.y];
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    // a point is dense exactly when its parent is set (k_b_dense_init gives
    // dense points an ancestor, the others -1, and unions only move roots to
    // smaller roots), so the parents answer both density tests without the
    // counts
    int *pr = par + B.base;
    const int pp = pr[p];
    if (pp < 0) return;
    // the recorded neighbours: -1 where there is none (phi mode records them too)
    int q[kSampleEdges], pq[kSampleEdges];
#pragma unroll
    for (int e = 0; e < kSampleEdges; ++e) q[e] = nb[kSampleEdges * (B.nbase + p) + e];
#pragma unroll
    for (int e = 0; e < kSampleEdges; ++e) pq[e] = q[e] >= 0 && q[e] < n ? pr[q[e]] : -1;
    // equal parents are one set, decided without reading the root's own entry
    // (which every point of a large component would read at once)
#pragma unroll
    for (int e = 0; e < kSampleEdges; ++e)
        if (pq[e] >= 0 && pq[e] != pp) uf_union(pr, p, q[e]);
}

__global__ void k_b_uf_compress(const BatchSub *__restrict__ subs, int n, const int *__restrict__ fit,
                                int *__restrict__ par) {
    if (fit && fit[blockIdx.y]) return;
    int *pr = par + subs[blockIdx.y].base;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || pr[i] < 0) return;
    // only the own entry is written, and once (uf_find shortens the entries it
    // passes: a late one of its writes could undo a root written here)
    int r = i;
    for (int p = ld_relaxed(&pr[r]); p != r; p = ld_relaxed(&pr[r])) r = p;
    st_relaxed(&pr[i], r);
}

// the parents in sorted order, for the full phase; zeroed sizes
__global__ void k_b_rootpos(const BatchSub *__restrict__ subs, int n, const int *__restrict__ par,
                            int *__restrict__ rootpos) {
    const BatchSub &B = subs[blockIdx.y];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    rootpos[B.base + i] = par[B.base + B.order[i]];
    B.csize[i] = 0;
}

// one block of 256 per subspace: the most frequent root among 256 evenly
// spaced points
__global__ void k_b_giant(const BatchSub *__restrict__ subs, int n, const int *__restrict__ fit,
                          const int *__restrict__ par, int *__restrict__ giant) {
    if (fit && fit[blockIdx.x]) return;
    __shared__ int roots[256];
    __shared__ int best_c[256];
    __shared__ int best_r[256];
    const int *pr = par + subs[blockIdx.x].base;
    const int t = threadIdx.x;
    const int p = (int) (((long long) t * n) / 256);
    roots[t] = p < n ? pr[p] : -1;
    __syncthreads();
    int r = roots[t], c = 0;
    if (r >= 0)
        for (int u = 0; u < 256; ++u) c += roots[u] == r;
    best_c[t] = c;
    best_r[t] = r;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (t < w && (best_c[t + w] > best_c[t] || (best_c[t + w] == best_c[t] && best_r[t + w] < best_r[t] &&
                                                    best_c[t + w] > 0))) {
            best_c[t] = best_c[t + w];
            best_r[t] = best_r[t + w];
        }
        __syncthreads();
    }
    if (t == 0) giant[blockIdx.x] = best_c[0] > 0 ? best_r[0] : -1;
}

// Full phase: every dense point outside the giant component links to all its
// dense neighbours.  Nearly all candidates are in the point's own set after the
// sample phase, so a step reads the roots of that phase first (rootpos, by
// sorted position, -1 where not dense: kLinkGroups groups of four per lane in
// flight), and only a group with a root of another set is tested on its ids,
// coordinates and cells (tested first, every candidate cost K + 2 loads:
// n=100,000 d=20 38.3 -> 34.2 ms a run, n=25,000 d=15 1.6 -> 1.2; one group in
// flight 36.1).  The staging of a query is what bounds it now.
// K > 0: every subspace of the launch has k = K.
constexpr int kLinkGroups = 4;
template <int K>
__global__ __launch_bounds__(kBlock) void k_b_link_full(const BatchSub *__restrict__ subs, int n,
                                                        const float *__restrict__ edge,
                                                        const int *__restrict__ rootpos, float s_star,
                                                        const int *__restrict__ giant, int *__restrict__ par) {
    constexpr int LPQ = kBLanes;
    extern __shared__ char smem[];
    const BatchSub &B = subs[blockIdx.y];
    const int k = B.S.k;
    float2 *sc;
    float *sy;
    int *qr;
    lds_layout(smem, k, sc, sy, qr);
    const int lq = threadIdx.x / LPQ, sub = threadIdx.x % LPQ;
    const int i = blockIdx.x * QPB + lq;
    const int *rts = rootpos + B.base;
    const int *ord = B.order;
    int *pr = par + B.base;
    const int r0 = i < n ? rts[i] : -1;  // the point's set after the sample phase
    const bool active = r0 >= 0 && r0 != giant[blockIdx.y];
    int *q = qr + lq * kRangeWords;
    // r0 stands for the point in every union: its parent is read while the
    // query is staged
    int rp = active ? uf_find(pr, r0) : -1;
    if (active) stage_query_b(B, edge, i, sub, s_star, sy + lq, sc + lq, QPB, q);
    if (!active) return;
    const float *qy = sy + lq;
    const float2 *qcl = sc + lq;
    const int total = q[18];
    if constexpr (K > 0) {
        // each lane four consecutive candidates of one run per group (the
        // groups of walk_vec)
        typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
        typedef int i4u __attribute__((ext_vector_type(4), aligned(4)));
        constexpr int U = 4, W = kLinkGroups;
        const uint32_t checked = (uint32_t) B.G.checkmask;
        const int gtotal = q[29];
        int r = 0, rgend = q[21];
        for (int g0 = 0; g0 < gtotal; g0 += W * LPQ) {
            int at[W], nv[W];
            i4u rt[W];
#pragma unroll
            for (int w = 0; w < W; ++w) {
                const int gw = g0 + w * LPQ + sub;
                const int g = min(gw, gtotal - 1);
                while (g >= rgend) {
                    ++r;
                    rgend = q[21 + r];
                }
                const int e0 = (g - q[20 + r]) << 2;
                nv[w] = gw < gtotal ? min(U, q[10 + r] - q[9 + r] - e0) : 0;
                at[w] = q[r] + e0;
                rt[w] = *reinterpret_cast<const i4u *>(rts + (uint32_t) at[w]);
            }
#pragma unroll
            for (int w = 0; w < W; ++w) {
                bool other[U], any = false;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    other[u] = (u < nv[w]) & (rt[w][u] >= 0) & (rt[w][u] != r0);
                    any |= other[u];
                }
                if (!any) continue;
                const int jj0 = at[w];
                const i4u id = *reinterpret_cast<const i4u *>(ord + (uint32_t) jj0);
                float acc[U] = {};
#pragma unroll
                for (int t = 0; t < K; ++t) {
                    const f4u y = *reinterpret_cast<const f4u *>(B.col[t] + (uint32_t) jj0);
                    const float qv = qy[t * QPB];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const float diff = qv - y[u];
                        const float sq = diff * diff;
                        acc[u] = acc[u] + sq;
                    }
                }
#pragma unroll
                for (int u = 0; u < U; ++u) other[u] &= acc[u] <= s_star;
                if (checked) cells_of_hits<U>(B, qcl, QPB, checked, jj0, other);
                // parents only move up to roots: a parent equal to p's root is p's set
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (!other[u] || pr[id[u]] == rp || uf_find(pr, id[u]) == rp) continue;
                    uf_union(pr, r0, id[u]);
                    rp = uf_find(pr, r0);
                }
            }
        }
    } else {
        int r = 0;
        for (int c = sub; c < total; c += LPQ) {
            const int jj = run_pos(q, c, r);
            float acc;
            if (rts[jj] < 0 || rts[jj] == r0 || !cand_test(B, qy, qcl, QPB, jj, s_star, acc)) continue;
            const int qq = ord[jj];
            // parents only move up to roots: a parent equal to p's root is p's set
            if (pr[qq] == rp || uf_find(pr, qq) == rp) continue;
            uf_union(pr, r0, qq);
            rp = uf_find(pr, r0);
        }
    }
}

__global__ void k_b_uf_flatten(const BatchSub *__restrict__ subs, int n, int *__restrict__ par) {
    const BatchSub &B = subs[blockIdx.y];
    int *pr = par + B.base;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    int c = -1;
    if (i < n && pr[i] >= 0) c = uf_find(pr, i);
    wave_add_by_key(B.csize, c, c >= 0);
    if (i < n) B.comp[i] = c;
}

// ------------------------------------------------------------ partition of every (tree, dimension) pair
// Only the weak-dense points and the
// paths are written; a path's origin keeps its "point of this tree" bit when
// the origin survives the weak-density prune of the group.
__global__ void k_b_part_count(const PartPair *__restrict__ pairs, const int *__restrict__ blk_off, int np,
                               const uint8_t *__restrict__ cellC, int n, int thr, int wbit) {
    __shared__ int h[4 * 256];
    const int j = seg_of(blk_off, np, blockIdx.x);
    const PartPair &A = pairs[j];
    const int blk = blockIdx.x - blk_off[j];
    const int G = A.G;
    const uint8_t *cm = cellC + (size_t) A.m * n;
    for (int t = threadIdx.x; t < 4 * G; t += blockDim.x) h[t] = 0;
    __syncthreads();
    if (blk < A.bp) {
        for (int u = 0; u < kPartPerThread; ++u) {
            const int i = (blk * kPartPerThread + u) * blockDim.x + threadIdx.x;
            if (i < A.nP && (!A.keep || A.keep[i])) {
                const int p = A.P[i];
                const int g = A.gid[cm[p]];
                atomicAdd(&h[g], 1);
                if (meets(A.weakcnt[p], thr, wbit)) atomicAdd(&h[G + g], 1);
            }
        }
    } else {
        for (int u = 0; u < kPartPerThread; ++u) {
            const int i = ((blk - A.bp) * kPartPerThread + u) * blockDim.x + threadIdx.x;
            if (i < A.nsp) {
                const dmask_t mk = mload(A.spm, i, A.mw) & dabove(A.m);
                if (mk) {
                    const int g = A.gid[cm[origin(A.spx[i])]];
                    atomicAdd(&h[2 * G + g], 1);
                    atomicAdd(&h[3 * G + g], dcount(mk));
                }
            }
        }
    }
    __syncthreads();
    // the paths' branch levels (the size of their prune's table) follow the cursors
    unsigned long long *levels = reinterpret_cast<unsigned long long *>(A.cnt + 6 * G);
    for (int t = threadIdx.x; t < 4 * G; t += blockDim.x) {
        if (!h[t]) continue;
        if (t < 3 * G)
            atomicAdd(&A.cnt[t], h[t]);
        else
            atomicAdd(&levels[t - 3 * G], (unsigned long long) h[t]);
    }
}

// Only the groups whose weak-dense points reach min_size become surviving
// trees; the lists of the others are never read, so they are not written (a
// pair without such a group does nothing).  Slots: LDS ranks within the block,
// then one global reservation per (block, group).  Each thread takes
// kPartPerThread elements, one block-width apart.
__global__ void k_b_part_scatter(const PartPair *__restrict__ pairs, const int *__restrict__ blk_off, int np,
                                 const uint8_t *__restrict__ cellC, int n, int thr, int wbit, int min_size) {
    __shared__ int base[3 * 256];
    __shared__ int lcnt[3 * 256];
    __shared__ int lres[3 * 256];
    __shared__ int any_pass;
    const int j = seg_of(blk_off, np, blockIdx.x);
    const PartPair &A = pairs[j];
    const int blk = blockIdx.x - blk_off[j];
    const int G = A.G;
    const uint8_t *cm = cellC + (size_t) A.m * n;
    if (threadIdx.x == 0) any_pass = 0;
    for (int t = threadIdx.x; t < 3 * G; t += blockDim.x) lcnt[t] = 0;
    __syncthreads();
    for (int g = threadIdx.x; g < G; g += blockDim.x)
        if (A.cnt[G + g] >= min_size) any_pass = 1;
    if (threadIdx.x < 3) {
        int acc = 0;
        for (int g = 0; g < G; ++g) {
            base[threadIdx.x * G + g] = acc;
            acc += A.cnt[threadIdx.x * G + g];
        }
    }
    __syncthreads();
    if (!any_pass) return;  // uniform over the block
    int *cur = A.cnt + 3 * G;
    const bool pts = blk < A.bp;
    int key[kPartPerThread], rnk[kPartPerThread], val[kPartPerThread];
    dmask_t mk[kPartPerThread];
    for (int u = 0; u < kPartPerThread; ++u) {
        key[u] = -1;
        rnk[u] = 0;
        val[u] = 0;
        mk[u] = 0;
        if (pts) {
            const int i = (blk * kPartPerThread + u) * blockDim.x + threadIdx.x;
            if (i < A.nP && (!A.keep || A.keep[i])) {
                const int p = A.P[i];
                const int g = A.gid[cm[p]];
                if (A.cnt[G + g] >= min_size && meets(A.weakcnt[p], thr, wbit)) {
                    key[u] = G + g;
                    val[u] = p;
                }
            }
        } else {
            const int i = ((blk - A.bp) * kPartPerThread + u) * blockDim.x + threadIdx.x;
            if (i < A.nsp) {
                mk[u] = mload(A.spm, i, A.mw) & dabove(A.m);
                const int xr = A.spx[i];
                const int xo = origin(xr);
                const int g = A.gid[cm[xo]];
                if (mk[u] && A.cnt[G + g] >= min_size) {
                    key[u] = 2 * G + g;
                    val[u] = (xr >= 0 && meets(A.weakcnt[xo], thr, wbit)) ? xo : ~xo;
                }
            }
        }
        if (key[u] >= 0) rnk[u] = atomicAdd(&lcnt[key[u]], 1);
    }
    __syncthreads();
    for (int t = threadIdx.x; t < 3 * G; t += blockDim.x)
        if (lcnt[t]) lres[t] = atomicAdd(&cur[t], lcnt[t]);
    __syncthreads();
    for (int u = 0; u < kPartPerThread; ++u) {
        if (key[u] < 0) continue;
        const int pos = base[key[u]] + lres[key[u]] + rnk[u];
        if (pts) {
            A.outW[pos] = val[u];
        } else {
            A.outx[pos] = val[u];
            mstore(A.outm, pos, mk[u], A.mw);
        }
    }
}

// ------------------------------------------------------------ path prune of every surviving tree
// A path (b, x) survives the prune when some surviving point w shares x's cells
// at every unrestricted level <= b; a path whose origin is in the tree (x >= 0)
// always does.  The prefixes asked for (a few per path whose origin is gone) go
// into an open-addressing table of (32 hash bits | origin), every point of the
// tree looks its own prefixes up and marks the ones it finds, and the paths
// keep their marked levels.  (The other way round, a table of every point's
// prefixes at every level, is 10 to 50 times larger and was bound by its
// scattered swaps: n=20,011 d=70 28.9 ms a run against 9.9.)  Every hit is
// confirmed on the cells.  Identity order: level t is dimension t.
constexpr uint32_t kMarked = 1u << 31;  // in the low word of a slot (n < 2^30)
constexpr uint32_t kOriginMask = (1u << 30) - 1;

// slot of the prefix of z through level t, or -1; e: its hash
__device__ __forceinline__ long long path_slot(const DevData &D, const PruneChild &P, uint64_t e, int z, int t,
                                               uint64_t &cur) {
    uint64_t slot = e & P.tmask;
    while (true) {
        cur = P.table[slot];
        if (cur == kEmpty) return -1;
        if ((cur >> 32) == (e >> 32) && same_prefix(D, P.smask, z, (int) ((uint32_t) cur & kOriginMask), t))
            return (long long) slot;
        slot = (slot + 1) & P.tmask;
    }
}

// f(t, hash) for every unrestricted level t of `want` in level order
template <class F>
__device__ __forceinline__ void for_prefixes(const DevData &D, dmask_t smask, int z, dmask_t want, F f) {
    uint64_t h = 0x243F6A8885A308D3ull;
    CellRow row{};
    for (int t = 0; t < D.d && want; ++t) {
        if (!(t & 15)) row = load_row(D, z, t);
        if (dhas(smask, t)) continue;
        h = mix64(h + row.at(t & 15) + 1);
        if (!dhas(want, t)) continue;
        want &= ~dbit(t);
        f(t, mix64(h ^ (0x9E3779B97F4A7C15ull * (uint64_t) (t + 1))));
    }
}

__global__ void k_b_path_insert(DevData D, const PruneChild *__restrict__ C, const int *__restrict__ blk_p, int nc) {
    const int c = seg_of(blk_p, nc, blockIdx.x);
    const PruneChild &P = C[c];
    const int i = (blockIdx.x - blk_p[c]) * blockDim.x + threadIdx.x;
    dmask_t m = 0;
    if (i < P.nsp && P.spx[i] < 0) m = mload(P.spm, i, P.mw) & ~P.smask;
    wave_or_mask(m, P.bits);
    if (!m) return;
    const int z = ~P.spx[i];
    for_prefixes(D, P.smask, z, m, [&](int t, uint64_t e) {
        const uint64_t entry = (e & 0xFFFFFFFF00000000ull) | (uint32_t) z;
        uint64_t slot = e & P.tmask;
        while (true) {
            // a slot is written once, by the swap from empty: a plain load that
            // still sees it empty is corrected by the failed swap, a full one is final
            uint64_t cur = P.table[slot];
            if (cur == kEmpty) {
                cur = atomicCAS((unsigned long long *) &P.table[slot], (unsigned long long) kEmpty,
                                (unsigned long long) entry);
                if (cur == kEmpty) break;
            }
            if ((cur >> 32) == (entry >> 32) && same_prefix(D, P.smask, z, (int) (uint32_t) cur, t)) break;
            slot = (slot + 1) & P.tmask;
        }
    });
}

__global__ void k_b_path_mark(DevData D, const PruneChild *__restrict__ C, const int *__restrict__ blk_w, int nc) {
    const int c = seg_of(blk_w, nc, blockIdx.x);
    const PruneChild &P = C[c];
    const int i = (blockIdx.x - blk_w[c]) * blockDim.x + threadIdx.x;
    if (i >= P.nW) return;
    const dmask_t need = *P.bits;
    if (!need) return;
    const int w = P.W[i];
    for_prefixes(D, P.smask, w, need, [&](int t, uint64_t e) {
        uint64_t cur;
        const long long at = path_slot(D, P, e, w, t, cur);
        // every marker writes the same word
        if (at >= 0 && !((uint32_t) cur & kMarked))
            reinterpret_cast<uint32_t *>(P.table + at)[0] = (uint32_t) cur | kMarked;
    });
}

__global__ void k_b_path_check(DevData D, const PruneChild *__restrict__ C, const int *__restrict__ blk_p, int nc) {
    const int c = seg_of(blk_p, nc, blockIdx.x);
    const PruneChild &P = C[c];
    const int i = (blockIdx.x - blk_p[c]) * blockDim.x + threadIdx.x;
    int x = 0;
    dmask_t m = 0;
    if (i < P.nsp) {
        x = P.spx[i];
        m = mload(P.spm, i, P.mw);
        if (x < 0) {
            dmask_t keep = 0;
            for_prefixes(D, P.smask, ~x, m, [&](int t, uint64_t e) {
                uint64_t cur;
                if (path_slot(D, P, e, ~x, t, cur) >= 0 && ((uint32_t) cur & kMarked)) keep |= dbit(t);
            });
            m = keep;
        }
    }
    const int slot = wave_slot(m != 0, P.nout);
    if (m != 0) {
        P.outx[slot] = x;
        mstore(P.outm, slot, m, P.mw);
    }
}

// ------------------------------------------------------------ phi in leaf order
// phi_S(p) exactly as the reference sums it: over p's neighbours in the order
// of the neighbourhood tree's leaves (rank_order: points sorted by their eps
// cells over all dimensions in tree level order, ties by id), float running
// sum with a double term (ClusteringCpu.cu:116-124).  One block per point:
// the block walks all points in that order, 256 at a time, finds the
// neighbours (candidate cells within one in every matched dimension of S,
// then the distance) and one thread adds their terms in order.
__global__ __launch_bounds__(kBlock) void k_b_phi_exact(DevData D, const BatchSub *__restrict__ subs,
                                                        const int2 *__restrict__ fb, const int *__restrict__ nfb,
                                                        int fbcap, const int *__restrict__ rank_order, float eps,
                                                        float s_star) {
    __shared__ double terms[kBlock];
    __shared__ int wcnt[kBlock / 64];
    __shared__ float qv[kMaxSubDims];
    __shared__ int qc[kMaxSubDims];
    const int count = min(*nfb, fbcap);
    const int n = D.n;
    const int lane = __lane_id(), wave = threadIdx.x / 64;
    for (int item = blockIdx.x; item < count; item += gridDim.x) {
        const int2 it = fb[item];
        const BatchSub &B = subs[it.x];
        const int p = it.y;
        const int k = B.S.k;
        if ((int) threadIdx.x < k) {
            const int s = B.S.dims[threadIdx.x];
            qv[threadIdx.x] = D.Xt[(size_t) s * n + p];
            qc[threadIdx.x] = D.cellE[(size_t) s * n + p];
        }
        __syncthreads();
        float sum = 0.0f;
        long long nterm = 0;
        for (int base = 0; base < n; base += kBlock) {
            const int rk = base + (int) threadIdx.x;
            bool hit = false;
            double term = 0.0;
            if (rk < n) {
                const int q = rank_order[rk];
                bool ok = q != p;
                for (int t = 0; t < k && ok; ++t) {
                    if (!((B.matchmask >> t) & 1ull)) continue;
                    const int de = (int) D.cellE[(size_t) B.S.dims[t] * n + q] - qc[t];
                    ok = de >= -1 && de <= 1;
                }
                if (ok) {
                    float acc = 0.0f;
                    for (int t = 0; t < k; ++t) {
                        const float diff = qv[t] - D.Xt[(size_t) B.S.dims[t] * n + q];
                        const float sq = diff * diff;
                        acc = acc + sq;
                    }
                    if (acc <= s_star) {
                        hit = true;
                        term = phi_term(acc, eps);
                    }
                }
            }
            const unsigned long long m = __ballot(hit);
            if (lane == 0) wcnt[wave] = __popcll(m);
            __syncthreads();
            int off0 = 0, tot = 0;
            for (int w = 0; w < kBlock / 64; ++w) {
                if (w < wave) off0 += wcnt[w];
                tot += wcnt[w];
            }
            if (hit) terms[off0 + __popcll(m & ((1ull << lane) - 1ull))] = term;
            __syncthreads();
            if (threadIdx.x == 0)
                for (int t = 0; t < tot; ++t) sum = (float) ((double) sum + terms[t]);
            nterm += tot;
            __syncthreads();
        }
        // the float sum bounds T within N 2^-22 (so T <= sum (1 + 2 N 2^-22)
        // while N 2^-22 <= 1/2), and the stored bound adds N 2^-22 once more
        const double rel = (double) nterm * (1.0 / 4194304.0);
        if (threadIdx.x == 0)
            B.cnt[p] = phi_code((sum >= B.phi_w ? 1 : 0) | (sum >= B.phi_d ? 2 : 0),
                                rel <= 0.25 ? (double) sum * (1.0 + 4.0 * rel) : -1.0);
        __syncthreads();
    }
}

// ------------------------------------------------------------ replay of pruneRedundancy and join
// The reference's depth-first order is replayed in stages: one launch per
// pass serves every step of a stage (the host groups the steps).  `list`
// holds the result-table rows whose subspace contains S (fixed once the
// expansion is done); a row counts while its nkept > 0, which the joins of
// earlier stages have set.  A tree is known by its index; tstamp[p] is the
// tree of S whose weak-dense points hold p.
//
// Both row walks (redundancy, join check) are planned in LDS: every block of
// a step reads a segment of up to kSegRows rows at once, cuts each row's walk
// into chunks of kChunk items and takes every nb-th chunk (nb: the step's
// blocks), so no block walks the rows one after another.
constexpr int kChunk = 2048;
constexpr int kSegRows = 1024;

struct RowPlan {
    int len[kSegRows];      // items of the row's walk (0: the row is not in the result)
    int pre[kSegRows + 1];  // chunks before each row
    uint8_t by_mem[kSegRows];
};

// loads rows [seg, seg + ns) of the list and their chunk prefix (of the items
// past the first `head`); returns the number of chunks.  by_mem: walk the row's
// members (else the tree's points, when nW is shorter; nW < 0 walks members
// always).  A row without a kept cluster of at least `floor` points is not walked.
__device__ int plan_rows(const Entry *__restrict__ E, const int *__restrict__ list, int seg, int ns, int nW, int head,
                         double floor, RowPlan &R, int *wtmp) {
    for (int i = threadIdx.x; i < ns; i += blockDim.x) {
        const Entry e = E[list[seg + i]];
        const bool bm = nW < 0 || e.nmem <= nW;
        R.len[i] = e.nkept > 0 && !(floor > (double) e.maxk) ? (bm ? e.nmem : nW) : 0;
        R.by_mem[i] = bm ? 1 : 0;
    }
    __syncthreads();
    // exclusive prefix of chunk counts: 4 rows per thread, then a block scan
    constexpr int PER = kSegRows / kBlock;
    int c[PER], sum = 0;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int i = threadIdx.x * PER + u;
        c[u] = i < ns ? (max(R.len[i] - head, 0) + kChunk - 1) / kChunk : 0;
        sum += c[u];
    }
    int incl = sum;
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(incl, o);
        if (__lane_id() >= o) incl += v;
    }
    if (__lane_id() == 63) wtmp[threadIdx.x / 64] = incl;
    __syncthreads();
    int before = 0, total = 0;
    for (int w = 0; w < kBlock / 64; ++w) {
        if (w < (int) threadIdx.x / 64) before += wtmp[w];
        total += wtmp[w];
    }
    int at = before + incl - sum;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int i = threadIdx.x * PER + u;
        if (i < ns) R.pre[i] = at;
        at += c[u];
    }
    if (threadIdx.x == 0) R.pre[ns] = total;
    __syncthreads();
    return total;
}

// row of chunk w: the last i with pre[i] <= w (rows without chunks share
// their successor's offset)
__device__ __forceinline__ int row_of(const RowPlan &R, int ns, int w) {
    int lo = 0, hi = ns;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (R.pre[mid] <= w)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// ---- the staged replay: every pass serves all steps of one stage
__device__ __forceinline__ int flag_cand(int J) { return -(2 + 3 * J); }
__device__ __forceinline__ int flag_drop(int J) { return -(3 + 3 * J); }
__device__ __forceinline__ int flag_fresh(int J) { return -(4 + 3 * J); }

// pruneRedundancy of every step with a tree (the step's own block range stands
// for the grid).  A row drops the tree when the tree touches it and no cluster
// touched is smaller than |T| r: a row whose largest kept cluster is smaller
// cannot and is left out (n=100,000 d=20: 20.7 -> 8.5 ms a run; n=25,000 d=15:
// 1.10 -> 0.58).  Of the others most that the tree touches show a
// smaller cluster among their first items: every row is probed first, a wave per
// row, and only the rows left over are walked on in chunks (n=100,000 d=20:
// 25.4 -> 20.7 ms, before rows were left out).
constexpr int kProbe = 256;
__global__ void k_rep_red_multi(const RepOp *__restrict__ ops, const int *__restrict__ blk_off, int nops,
                                const Entry *__restrict__ E, float r, int *__restrict__ keepv) {
    __shared__ RowPlan R;
    __shared__ int wtmp[kBlock / 64];
    __shared__ int skip;
    __shared__ bool last;
    const int o = seg_of(blk_off, nops, blockIdx.x);
    const RepOp &Op = ops[o];
    const int nb = blk_off[o + 1] - blk_off[o], bi = blockIdx.x - blk_off[o];
    const int nlist = Op.nlist, nW = Op.nW, tree = Op.tree;
    const int *list = Op.list;
    int *rowflag = Op.rowflag;
    const double lhs = (double) ((float) nW * r);
    // item t of a row: (touch, small)
    auto item = [&](const Entry &e, bool by_mem, int t, bool &touch, bool &small) {
        if (by_mem) {
            const int q = e.mem[t];
            if (Op.tstamp[q] == tree) {
                touch = true;
                small |= lhs > (double) e.csize[e.comp[q]];
            }
        } else {
            const int K = e.comp[Op.W[t]];
            if (K >= 0 && e.inres[K]) {
                touch = true;
                small |= lhs > (double) e.csize[K];
            }
        }
    };
    for (int seg = 0; seg < nlist; seg += kSegRows) {
        const int ns = min(kSegRows, nlist - seg);
        const int total = plan_rows(E, list, seg, ns, nW, kProbe, lhs, R, wtmp);
        constexpr int W = kBlock / 64;
        for (int i = bi * W + (int) (threadIdx.x / 64); i < ns; i += nb * W) {
            const int len = min(R.len[i], kProbe);
            if (len == 0) continue;
            const Entry e = E[list[seg + i]];
            const bool by_mem = R.by_mem[i];
            bool touch = false, small = false;
            for (int t = __lane_id(); t < len; t += 64) item(e, by_mem, t, touch, small);
            const bool any_touch = __any(touch), any_small = __any(small);
            if (__lane_id() == 0) {
                if (any_touch) st_relaxed(&rowflag[2 * (seg + i)], 1);
                if (any_small) st_relaxed(&rowflag[2 * (seg + i) + 1], 1);
            }
        }
        __syncthreads();
        for (int w = bi; w < total; w += nb) {
            const int i = row_of(R, ns, w);
            const int h = seg + i;
            if (threadIdx.x == 0) skip = ld_relaxed(&rowflag[2 * h + 1]);
            __syncthreads();
            const bool sk = skip != 0;
            __syncthreads();
            if (sk) continue;
            const Entry e = E[list[h]];
            const bool by_mem = R.by_mem[i];
            const int t0 = kProbe + (w - R.pre[i]) * kChunk, t1 = min(R.len[i], t0 + kChunk);
            bool touch = false, small = false;
            for (int t = t0 + threadIdx.x; t < t1; t += blockDim.x) item(e, by_mem, t, touch, small);
            touch = __syncthreads_or(touch);
            small = __syncthreads_or(small);
            if (threadIdx.x == 0) {
                if (touch) st_relaxed(&rowflag[2 * h], 1);
                if (small) st_relaxed(&rowflag[2 * h + 1], 1);
            }
        }
        __syncthreads();
    }
    __threadfence();
    if (threadIdx.x == 0) last = atomicAdd(Op.done, 1u) == (unsigned) nb - 1;
    __syncthreads();
    if (last) {
        __threadfence();
        int drop = 0;
        for (int h = threadIdx.x; h < nlist; h += blockDim.x) {
            const int t = ld_relaxed(&rowflag[2 * h]), sm = ld_relaxed(&rowflag[2 * h + 1]);
            drop |= (t && !sm) ? 1 : 0;
        }
        drop = __syncthreads_or(drop);
        if (threadIdx.x == 0) keepv[tree] = drop ? 0 : 1;
    }
}

// candidates of every join step: the components (of at least min_size
// points) of the points of its kept trees; one list entry per component
__global__ void k_rep_cand_multi(const RepOp *__restrict__ ops, const int *__restrict__ blk_off, int nops,
                                 const int *__restrict__ keepv, int min_size, int n) {
    const int o = seg_of(blk_off, nops, blockIdx.x);
    const RepOp &Op = ops[o];
    const int i = (blockIdx.x - blk_off[o]) * blockDim.x + threadIdx.x;
    int K = -1;
    if (Op.kind == 0) {
        if (i < Op.nW && keepv[Op.tree]) K = Op.comp[Op.W[i]];
    } else if (i < n) {
        const int t = Op.tstamp[i];
        if (t >= Op.t_lo && t < Op.t_hi && keepv[t]) K = Op.comp[i];
    }
    const int cj = flag_cand(Op.J);
    bool want = K >= 0 && Op.csize[K] >= min_size && Op.flag[K] != cj;
    // one claim per distinct component in the wave
    unsigned long long todo = __ballot(want);
    while (todo) {
        const int leader = __ffsll((long long) todo) - 1;
        const int lk = __shfl(K, leader);
        todo &= ~__ballot(want && K == lk);
        if (__lane_id() == leader) {
            const int old = atomicExch(&Op.flag[lk], cj);
            if (old != cj) {
                const int at = atomicAdd(&Op.words[0], 1);
                if (at < Op.ccap) Op.clist[at] = lk;
            }
        }
    }
}

// a candidate K is dropped when one of its points lies in a result cluster of
// a superspace H larger than |K| * r
__global__ void k_rep_check_multi(const RepOp *__restrict__ ops, const int *__restrict__ blk_off, int nops,
                                  const Entry *__restrict__ E, float r) {
    __shared__ RowPlan R;
    __shared__ int wtmp[kBlock / 64];
    const int o = seg_of(blk_off, nops, blockIdx.x);
    const RepOp &Op = ops[o];
    if (ld_relaxed(&Op.words[0]) == 0) return;  // no candidate (uniform over the step's blocks)
    const int nb = blk_off[o + 1] - blk_off[o], bi = blockIdx.x - blk_off[o];
    const int cj = flag_cand(Op.J), dj = flag_drop(Op.J);
    for (int seg = 0; seg < Op.nlist; seg += kSegRows) {
        const int ns = min(kSegRows, Op.nlist - seg);
        const int total = plan_rows(E, Op.list, seg, ns, -1, 0, 0.0, R, wtmp);
        for (int w = bi; w < total; w += nb) {
            const int i = row_of(R, ns, w);
            const Entry e = E[Op.list[seg + i]];
            const int t0 = (w - R.pre[i]) * kChunk, t1 = min(R.len[i], t0 + kChunk);
            for (int t = t0 + threadIdx.x; t < t1; t += blockDim.x) {
                const int q = e.mem[t];
                const int K = Op.comp[q];
                if (K < 0 || Op.flag[K] != cj) continue;
                if ((float) Op.csize[K] * r < (float) e.csize[e.comp[q]]) Op.flag[K] = dj;
            }
        }
        __syncthreads();
    }
}

// the surviving candidates of every join step join the result of its
// subspace (one block per step)
__global__ void k_rep_apply_multi(const RepOp *__restrict__ ops, Entry *__restrict__ E) {
    __shared__ int wtmp[kBlock / 64], wmax[kBlock / 64];
    const RepOp &Op = ops[blockIdx.x];
    if (Op.kind == 1) return;
    const int nc = min(Op.words[0], Op.ccap);
    const int cj = flag_cand(Op.J), fj = flag_fresh(Op.J);
    int added = 0, most = 0;
    for (int k = threadIdx.x; k < nc; k += blockDim.x) {
        const int K = Op.clist[k];
        if (Op.flag[K] == cj && !Op.inres[K]) {
            Op.inres[K] = 1;
            Op.flag[K] = fj;
            ++added;
            most = max(most, Op.csize[K]);
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        added += __shfl_down(added, o);
        most = max(most, __shfl_down(most, o));
    }
    if (__lane_id() == 0) {
        wtmp[threadIdx.x / 64] = added;
        wmax[threadIdx.x / 64] = most;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int tot = 0;
        for (int w = 0; w < kBlock / 64; ++w) {
            tot += wtmp[w];
            most = max(most, wmax[w]);
        }
        if (tot) {
            E[Op.entry].nkept += tot;
            E[Op.entry].maxk = max(E[Op.entry].maxk, most);
        }
        Op.words[1] = tot;
    }
}

constexpr int kMemPerBlock = 1024;

// members of the newly joined clusters of every join step
__global__ void k_rep_members_multi(const RepOp *__restrict__ ops, const int *__restrict__ blk_off, int nops,
                                    Entry *__restrict__ E, int n) {
    __shared__ int wcount[kBlock / 64];
    __shared__ int base;
    const int o = seg_of(blk_off, nops, blockIdx.x);
    const RepOp &Op = ops[o];
    if (Op.words[1] == 0) return;  // nothing joined (uniform over the step's blocks)
    const int fj = flag_fresh(Op.J);
    constexpr int PER = kMemPerBlock / kBlock;
    const int i0 = (blockIdx.x - blk_off[o]) * kMemPerBlock;
    bool in[PER];
    int mine = 0;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int i = i0 + u * kBlock + threadIdx.x;
        bool f = false;
        if (i < n) {
            const int K = Op.comp[i];
            f = K >= 0 && Op.flag[K] == fj;
        }
        in[u] = f;
        mine += f ? 1 : 0;
    }
    int incl = mine;
    for (int d = 1; d < 64; d <<= 1) {
        const int v = __shfl_up(incl, d);
        if (__lane_id() >= d) incl += v;
    }
    if (__lane_id() == 63) wcount[threadIdx.x / 64] = incl;
    __syncthreads();
    int before = 0, total = 0;
    for (int w = 0; w < kBlock / 64; ++w) {
        if (w < (int) threadIdx.x / 64) before += wcount[w];
        total += wcount[w];
    }
    if (threadIdx.x == 0) base = total > 0 ? atomicAdd(&E[Op.entry].nmem, total) : 0;
    __syncthreads();
    int slot = base + before + incl - mine;
    int *mem = E[Op.entry].mem;
#pragma unroll
    for (int u = 0; u < PER; ++u)
        if (in[u]) mem[slot++] = i0 + u * kBlock + threadIdx.x;
}

// ------------------------------------------------------------ small helpers
__global__ void k_b_copy(const CopySeg *__restrict__ segs, const int *__restrict__ blk_off, int ns) {
    const int s = seg_of(blk_off, ns, blockIdx.x);
    const CopySeg S = segs[s];
    const int i = (blockIdx.x - blk_off[s]) * blockDim.x + threadIdx.x;
    if (i >= S.len) return;
    const int v = S.src[i];
    if (S.pad < 0)
        S.dst[i] = v;
    else
        S.dst[v] = S.pad;
}

template <class T>
__global__ void k_b_fill(T *p, T v, size_t count) {
    fill_span(p, v, count);
}

}  // namespace

#define LAUNCH(kernel, grid, block, lds, st, ...) hipLaunchKernelGGL(kernel, grid, block, lds, st, __VA_ARGS__)

static_assert(kBlockThreads == kBlock && kQueriesPerBlock == QPB, "launch geometry constants disagree");

static unsigned query_blocks_n(int n) { return (unsigned) ((n + QPB - 1) / QPB); }
static size_t count_lds(int kmax) {
    return (sizeof(float2) + sizeof(float)) * QPB * (size_t) (kmax > 0 ? kmax : 1) + sizeof(int) * QPB * kRangeWords;
}

hipError_t launch_b_root(const dmask_t *nearm, int n, int *P, int *outx, uint64_t *outm, int mw, int *nout, int C,
                         float *edge, hipStream_t st) {
    LAUNCH(k_b_root, dim3(blocks_for((size_t) std::max(n, C + 3))), dim3(kBlock), 0, st, nearm, n, P, outx, outm, mw,
           nout, C, edge);
    return hipGetLastError();
}

hipError_t launch_b_flags(const FlagTree *T, const int *blk_off, int nt, int nblk, const uint8_t *cellC, int n,
                          int cells, int *flags, hipStream_t st) {
    if (nblk <= 0) return hipSuccess;
    LAUNCH(k_b_flags, dim3(nblk), dim3(kBlock), 0, st, T, blk_off, nt, cellC, n, cells, flags);
    return hipGetLastError();
}

hipError_t launch_b_sort(const DevData &D, const SortJob *jobs, int njob, int hmiss, int max_cell, int *keys,
                         int *rank, int *hist, int *off, void *scan_temp, size_t scan_bytes, hipStream_t st) {
    if (njob <= 0) return hipSuccess;
    const int nscan = hmiss + 1;  // the scan ends with the total
    LAUNCH(k_b_fill<int>, dim3(fill_blocks((size_t) nscan, sizeof(int))), dim3(kBlock), 0, st, hist, 0, (size_t) nscan);
    LAUNCH(k_b_keys, dim3(blocks_for(D.n), njob), dim3(kBlock), 0, st, D, jobs, keys, rank, hist);
    hipError_t e = launch_exclusive_sum(scan_temp, scan_bytes, hist, off, nscan, st);
    if (e != hipSuccess) return e;
    const unsigned span = blocks_for((size_t) std::max(D.n, max_cell + 1));
    LAUNCH(k_b_scatter, dim3(span, njob), dim3(kBlock), 0, st, D.n, jobs, keys, rank, off);
    return hipGetLastError();
}

hipError_t launch_b_gather(const ColJob *jobs, int njob, int n, hipStream_t st) {
    if (njob <= 0) return hipSuccess;
    const int nblk = (n + kBlock * kGatherItems - 1) / (kBlock * kGatherItems);
    LAUNCH(k_b_gather, dim3((unsigned) nblk * (unsigned) njob), dim3(kBlock), 0, st, jobs, n, nblk);
    return hipGetLastError();
}

// Ordered compaction of the query flags (one byte per sorted position, 0 or
// 1) into the positions that are set: a count per tile of 4,096 flags, an
// exclusive scan of the tile counts, and a write pass that ranks each lane's
// 16 flags inside its tile.  Every lane reads its flags as one 16-byte load;
// the flag array is padded to a multiple of 16 bytes and bytes at or past nb
// are ignored.
constexpr int kFlagsPerLane = 16;
constexpr int kFlagTile = kBlock * kFlagsPerLane;

__device__ __forceinline__ int set_bytes(uint32_t w) {
    w |= w >> 4;  // bit 0 of each byte: the OR of the byte's bits
    w |= w >> 2;
    w |= w >> 1;
    return __builtin_popcount(w & 0x01010101u);
}

__device__ __forceinline__ uint4 lane_flags(const uint8_t *__restrict__ qflag, size_t at, size_t nb) {
    if (at >= nb) return make_uint4(0, 0, 0, 0);
    uint4 v = *reinterpret_cast<const uint4 *>(qflag + at);
    if (at + kFlagsPerLane > nb) {
        uint32_t w[4] = {v.x, v.y, v.z, v.w};
        for (int q = 0; q < 4; ++q)
            for (int c = 0; c < 4; ++c)
                if (at + 4 * q + c >= nb) w[q] &= ~(0xffu << (8 * c));
        v = make_uint4(w[0], w[1], w[2], w[3]);
    }
    return v;
}

__global__ void __launch_bounds__(kBlock) k_b_flag_count(const uint8_t *__restrict__ qflag, size_t nb, int ntile,
                                                          int *__restrict__ tcnt) {
    __shared__ int wsum[kBlock / 64];
    const size_t at = ((size_t) blockIdx.x * kBlock + threadIdx.x) * kFlagsPerLane;
    const uint4 v = lane_flags(qflag, at, nb);
    int c = set_bytes(v.x) + set_bytes(v.y) + set_bytes(v.z) + set_bytes(v.w);
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
    if (__lane_id() == 0) wsum[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        int t = 0;
        for (int q = 0; q < kBlock / 64; ++q) t += wsum[q];
        tcnt[blockIdx.x] = t;
        if (blockIdx.x == 0) tcnt[ntile] = 0;  // the scan's last entry is the total
    }
}

__global__ void __launch_bounds__(kBlock) k_b_flag_write(const uint8_t *__restrict__ qflag, size_t nb,
                                                          const int *__restrict__ toff, int ntile,
                                                          int *__restrict__ qlist, int *__restrict__ nsel, int n,
                                                          int *__restrict__ qstart) {
    __shared__ int wsum[kBlock / 64];
    const size_t at = ((size_t) blockIdx.x * kBlock + threadIdx.x) * kFlagsPerLane;
    const uint4 v = lane_flags(qflag, at, nb);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    int m[4], c = 0;
    for (int q = 0; q < 4; ++q) {
        uint32_t x = w[q];
        x |= x >> 4;
        x |= x >> 2;
        x |= x >> 1;
        m[q] = (int) (x & 0x01010101u);
        c += __builtin_popcount((uint32_t) m[q]);
    }
    const int lane = __lane_id();
    int x = c;  // inclusive scan over the wave
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) wsum[threadIdx.x >> 6] = x;
    __syncthreads();
    int o = toff[blockIdx.x] + x - c;
    for (int q = 0; q < (int) (threadIdx.x >> 6); ++q) o += wsum[q];
    // qstart[b]: queries before position b * n (the first of subspace b)
    if (qstart && at < nb) {
        for (size_t b = (at + n - 1) / n; b * n < at + kFlagsPerLane && b * n < nb; ++b) {
            const int off = (int) (b * n - at);
            int before = o;
            for (int q = 0; q < 4; ++q)
                if (4 * q < off)
                    before += __builtin_popcount((uint32_t) m[q] & (off - 4 * q >= 4 ? ~0u : (1u << (8 * (off - 4 * q))) - 1u));
            qstart[b] = before;
        }
    }
    for (int q = 0; q < 4; ++q) {
        uint32_t mm = (uint32_t) m[q];
        while (mm) {
            const int bit = __builtin_ctz(mm);
            qlist[o++] = (int) (at + 4 * q + (bit >> 3));
            mm &= mm - 1;
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *nsel = toff[ntile];
        if (qstart) qstart[nb / n] = toff[ntile];
    }
}

static int flag_tiles(size_t items) { return (int) ((items + kFlagTile - 1) / kFlagTile); }

static size_t align256(size_t b) { return (b + 255) & ~(size_t) 255; }

size_t select_temp_bytes(int items) {
    const int nt = flag_tiles((size_t) std::max(items, 1));
    return 2 * align256((size_t) (nt + 1) * sizeof(int)) + align256(scan_temp_bytes(nt + 1));
}

hipError_t launch_flag_compact(const uint8_t *flags, size_t nb, void *temp, size_t temp_bytes, int *out, int *nsel,
                               int n, int *qstart, hipStream_t st) {
    const int nt = flag_tiles(nb);
    const size_t cnt_bytes = align256((size_t) (nt + 1) * sizeof(int));
    char *base = static_cast<char *>(temp);
    int *tcnt = reinterpret_cast<int *>(base);
    int *toff = reinterpret_cast<int *>(base + cnt_bytes);
    LAUNCH(k_b_flag_count, dim3(nt), dim3(kBlock), 0, st, flags, nb, nt, tcnt);
    hipError_t e = launch_exclusive_sum(base + 2 * cnt_bytes, temp_bytes - 2 * cnt_bytes, tcnt, toff, nt + 1, st);
    if (e != hipSuccess) return e;
    LAUNCH(k_b_flag_write, dim3(nt), dim3(kBlock), 0, st, flags, nb, toff, nt, out, nsel, n,
           qstart);
    return hipGetLastError();
}

hipError_t launch_b_queries(const BatchSub *subs, int nsub, int n, const QuerySeg *segs, const int *blk_off,
                            int nseg, int nblk, const BatchIndex &X, int *seg, hipStream_t st) {
    if (nsub <= 0) return hipSuccess;
    const size_t nb = (size_t) nsub * n;
    if (nblk > 0)
        LAUNCH(k_b_qmark, dim3(nblk), dim3(kBlock), 0, st, subs, segs, blk_off, nseg, X.qflag, seg);
    return launch_flag_compact(X.qflag, nb, X.select_temp, X.select_bytes, X.qlist, X.nsel, n, X.qstart, st);
}

template <int K>
static void launch_count_k(const BatchSub *subs, int nsub, const int *blk_off, int nblk, int n, size_t lds,
                           const BatchIndex &X, float s_star, float eps, double phirel, bool phi,
                           unsigned long long *stat, hipStream_t st) {
    if (blk_off) {
        if (phi)
            LAUNCH((k_b_count<true, true, K>), dim3(nblk), dim3(kBlock), lds, st, subs, blk_off, nsub, n,
                   X.edge, X.qlist, X.qstart, s_star, eps, phirel, X.nb, X.fb, X.nfb, X.fbcap, stat);
        else
            LAUNCH((k_b_count<true, false, K>), dim3(nblk), dim3(kBlock), lds, st, subs, blk_off, nsub, n,
                   X.edge, X.qlist, X.qstart, s_star, eps, phirel, X.nb, X.fb, X.nfb, X.fbcap, stat);
    } else {
        const dim3 grid(query_blocks_n(n), nsub);
        if (phi)
            LAUNCH((k_b_count<false, true, K>), grid, dim3(kBlock), lds, st, subs, (const int *) nullptr, nsub, n,
                   X.edge, X.qlist, X.qstart, s_star, eps, phirel, X.nb, X.fb, X.nfb,
                   X.fbcap, stat);
        else
            LAUNCH((k_b_count<false, false, K>), grid, dim3(kBlock), lds, st, subs, (const int *) nullptr, nsub, n,
                   X.edge, X.qlist, X.qstart, s_star, eps, phirel, X.nb, X.fb, X.nfb,
                   X.fbcap, stat);
    }
}

hipError_t launch_phi_exact(const DevData &D, const BatchSub *sub, const int2 *fb, const int *nfb, int fbcap,
                            const int *rank_order, float eps, float s_star, hipStream_t st) {
    LAUNCH(k_b_phi_exact, dim3(1024), dim3(kBlock), 0, st, D, sub, fb, nfb, fbcap, rank_order, eps, s_star);
    return hipGetLastError();
}

hipError_t launch_b_count(const BatchSub *subs, int nsub, const int *blk_off, int nblk, int n, int kmax, int kfast,
                          const BatchIndex &X, float s_star, float eps, bool phi, bool phi_all_exact,
                          const DevData &D, const int *rank_order, unsigned long long *stat, const KernelTimer &tm,
                          hipStream_t st) {
    // phi_all_exact: every point goes through the leaf-order recomputation (a test hook)
    const double phirel = phi_all_exact ? 1e30 : kPhiRelDefault;
    if (nsub <= 0) return hipSuccess;
    if (blk_off && nblk <= 0) return hipSuccess;
    if (phi) LAUNCH(k_b_fill<int>, dim3(1), dim3(kBlock), 0, st, X.nfb, 0, (size_t) 1);
    if (tm.start) (void) hipEventRecord(tm.start, st);
    const size_t lds = count_lds(kmax);
    switch (kfast) {
    case 1: launch_count_k<1>(subs, nsub, blk_off, nblk, n, lds, X, s_star, eps, phirel, phi, stat, st); break;
    case 2: launch_count_k<2>(subs, nsub, blk_off, nblk, n, lds, X, s_star, eps, phirel, phi, stat, st); break;
    case 3: launch_count_k<3>(subs, nsub, blk_off, nblk, n, lds, X, s_star, eps, phirel, phi, stat, st); break;
    case 4: launch_count_k<4>(subs, nsub, blk_off, nblk, n, lds, X, s_star, eps, phirel, phi, stat, st); break;
    case 5: launch_count_k<5>(subs, nsub, blk_off, nblk, n, lds, X, s_star, eps, phirel, phi, stat, st); break;
    case 6: launch_count_k<6>(subs, nsub, blk_off, nblk, n, lds, X, s_star, eps, phirel, phi, stat, st); break;
    case 7: launch_count_k<7>(subs, nsub, blk_off, nblk, n, lds, X, s_star, eps, phirel, phi, stat, st); break;
    case 8: launch_count_k<8>(subs, nsub, blk_off, nblk, n, lds, X, s_star, eps, phirel, phi, stat, st); break;
    default: launch_count_k<0>(subs, nsub, blk_off, nblk, n, lds, X, s_star, eps, phirel, phi, stat, st); break;
    }
    if (tm.stop) (void) hipEventRecord(tm.stop, st);
    if (phi)
        LAUNCH(k_b_phi_exact, dim3(1024), dim3(kBlock), 0, st, D, subs, X.fb, X.nfb, X.fbcap, rank_order, eps, s_star);
    return hipGetLastError();
}

template <bool PHI, int K>
static void launch_fan_width(int width, dim3 grid, hipStream_t st, const BatchSub *groups, const FanJob *jobs,
                             const int *blk_off, int njob, const FanTable &T, const DevData &D, const BatchIndex &X,
                             float s_star, float eps, double phirel, int cap, float phi_w, float phi_d,
                             unsigned long long *stat) {
#define FAN(CW, NC)                                                                                                    \
    LAUNCH((k_b_fan<PHI, K, CW, NC>), grid, dim3(kBlock), 0, st, groups, jobs, blk_off, njob, T, D.d, D.X, X.edge,    \
           X.qlist, X.qstart, s_star, eps, phirel, cap, phi_w, phi_d, X.nb, X.fb, X.nfb, X.fbcap, stat)
    switch (width) {
    case 4: FAN(4, 1); break;
    case 8: FAN(8, 1); break;
    case 16: FAN(8, 2); break;
    case 32: FAN(16, 2); break;
    default: FAN(16, 4); break;
    }
#undef FAN
}

hipError_t launch_b_fan(const BatchSub *groups, const FanJob *jobs, const int *blk_off, int njob, int nblk, int width,
                        int kS, const FanTable &T, const BatchIndex &X, float s_star, float eps, bool phi,
                        bool phi_all_exact, int cap, float phi_w, float phi_d, const DevData &D,
                        unsigned long long *stat, hipStream_t st) {
    if (njob <= 0 || nblk <= 0) return hipSuccess;
    if (kS < 1 || kS > kMaxFastK || width > kFanMost) return hipErrorInvalidValue;
    const double phirel = phi_all_exact ? 1e30 : kPhiRelDefault;
#define FAN_K(K)                                                                                                       \
    case K:                                                                                                            \
        if (phi)                                                                                                       \
            launch_fan_width<true, K>(width, dim3(nblk), st, groups, jobs, blk_off, njob, T, D, X, s_star, eps,       \
                                      phirel, cap, phi_w, phi_d, stat);                                                \
        else                                                                                                           \
            launch_fan_width<false, K>(width, dim3(nblk), st, groups, jobs, blk_off, njob, T, D, X, s_star, eps,      \
                                       phirel, cap, phi_w, phi_d, stat);                                               \
        break
    switch (kS) {
        FAN_K(1);
        FAN_K(2);
        FAN_K(3);
        FAN_K(4);
        FAN_K(5);
        FAN_K(6);
        FAN_K(7);
        FAN_K(8);
    }
#undef FAN_K
    return hipGetLastError();
}

hipError_t launch_b_components(const BatchSub *subs, int nsub, int n, int kmax, int kfast, const BatchIndex &X,
                               float s_star, hipStream_t st) {
    if (nsub <= 0) return hipSuccess;
    // In LDS (one block per subspace) while one block's pass over a subspace is
    // shorter than the swaps of all blocks on global parents.  Whole runs, d=8,
    // about 100 subspaces, LDS against global: n=39,936 5.9 / 6.7 ms, 60,000
    // 8.6 / 10.4, 100,000 18.9 / 22.6, 150,000 33.2 / 38.7, 200,000 57.7 / 57.3,
    // 300,000 108.8 / 103.2
    const bool lds_pass = n <= 4 * kUfCap;
    const int *fit = lds_pass ? X.fit : nullptr;
    const dim3 all(blocks_for(n), nsub);
    if (n > kUfCap) {
        LAUNCH(k_b_dense_init, all, dim3(kBlock), 0, st, subs, n, X.nb, X.par);
        LAUNCH(k_b_uf_compress, all, dim3(kBlock), 0, st, subs, n, (const int *) nullptr, X.par);
    }
    if (lds_pass)
        LAUNCH(k_b_sample, dim3(nsub), dim3(kUfThreads), 0, st, subs, n, X.nb, X.rootpos, X.par, X.giant, X.fit);
    if (n > kUfCap) {
        LAUNCH(k_b_link_sample, all, dim3(kBlock), 0, st, subs, n, X.nb, fit, X.par);
        LAUNCH(k_b_uf_compress, all, dim3(kBlock), 0, st, subs, n, fit, X.par);
        LAUNCH(k_b_rootpos, all, dim3(kBlock), 0, st, subs, n, X.par, X.rootpos);
        LAUNCH(k_b_giant, dim3(nsub), dim3(256), 0, st, subs, n, fit, X.par, X.giant);
    }
    const dim3 grid(query_blocks_n(n), nsub);
    const size_t lds = count_lds(kmax);
#define LINK_FULL(K)                                                                                                   \
    LAUNCH(k_b_link_full<K>, grid, dim3(kBlock), lds, st, subs, n, X.edge, X.rootpos,      \
           s_star, X.giant, X.par)
    switch (kfast) {
    case 1: LINK_FULL(1); break;
    case 2: LINK_FULL(2); break;
    case 3: LINK_FULL(3); break;
    case 4: LINK_FULL(4); break;
    case 5: LINK_FULL(5); break;
    case 6: LINK_FULL(6); break;
    case 7: LINK_FULL(7); break;
    case 8: LINK_FULL(8); break;
    default: LINK_FULL(0); break;
    }
#undef LINK_FULL
    LAUNCH(k_b_uf_flatten, dim3(blocks_for(n), nsub), dim3(kBlock), 0, st, subs, n, X.par);
    return hipGetLastError();
}

hipError_t launch_b_partition(const PartPair *pairs, const int *blk_off, int npairs, int nblk, const uint8_t *cellC,
                              int n, int thr, int wbit, int min_size, hipStream_t st) {
    if (nblk <= 0) return hipSuccess;
    LAUNCH(k_b_part_count, dim3(nblk), dim3(kBlock), 0, st, pairs, blk_off, npairs, cellC, n, thr, wbit);
    LAUNCH(k_b_part_scatter, dim3(nblk), dim3(kBlock), 0, st, pairs, blk_off, npairs, cellC, n, thr, wbit, min_size);
    return hipGetLastError();
}

hipError_t launch_b_prune(const DevData &D, const PruneChild *C, int nc, const int *blk_w, int nblk_w,
                          const int *blk_p, int nblk_p, hipStream_t st) {
    if (nc <= 0 || nblk_p <= 0) return hipSuccess;
    LAUNCH(k_b_path_insert, dim3(nblk_p), dim3(kBlock), 0, st, D, C, blk_p, nc);
    if (nblk_w > 0) LAUNCH(k_b_path_mark, dim3(nblk_w), dim3(kBlock), 0, st, D, C, blk_w, nc);
    LAUNCH(k_b_path_check, dim3(nblk_p), dim3(kBlock), 0, st, D, C, blk_p, nc);
    return hipGetLastError();
}

hipError_t launch_b_copy(const CopySeg *segs, const int *blk_off, int nseg, int nblk, hipStream_t st) {
    if (nblk <= 0) return hipSuccess;
    LAUNCH(k_b_copy, dim3(nblk), dim3(kBlock), 0, st, segs, blk_off, nseg);
    return hipGetLastError();
}

int rep_red_blocks(int nlist, int nW) { return std::max(1, std::min(nlist + nW / kChunk, 256)); }
int rep_check_blocks(int nlist, int n) { return nlist > 0 ? std::min(nlist + n / kChunk, 256) : 0; }
int rep_mem_blocks(int n) { return (n + kMemPerBlock - 1) / kMemPerBlock; }

hipError_t launch_rep_stage(const RepOp *ops, int nops, const int *blk_red, int nblk_red, const int *blk_cand,
                            int nblk_cand, const int *blk_chk, int nblk_chk, const int *blk_mem, int nblk_mem,
                            Entry *E, float r, int min_size, int n, int *keepv, hipStream_t st) {
    if (nops <= 0) return hipSuccess;
    if (nblk_red > 0) LAUNCH(k_rep_red_multi, dim3(nblk_red), dim3(kBlock), 0, st, ops, blk_red, nops, E, r, keepv);
    if (nblk_cand > 0)
        LAUNCH(k_rep_cand_multi, dim3(nblk_cand), dim3(kBlock), 0, st, ops, blk_cand, nops, keepv, min_size, n);
    if (nblk_chk > 0) LAUNCH(k_rep_check_multi, dim3(nblk_chk), dim3(kBlock), 0, st, ops, blk_chk, nops, E, r);
    LAUNCH(k_rep_apply_multi, dim3(nops), dim3(kBlock), 0, st, ops, E);
    if (nblk_mem > 0) LAUNCH(k_rep_members_multi, dim3(nblk_mem), dim3(kBlock), 0, st, ops, blk_mem, nops, E, n);
    return hipGetLastError();
}

}  // namespace inscy
