// HIP kernels of the MI355X INSCY engine (gfx950, wave64).
//
// Everything here is integer/byte streaming work plus one FP32 distance loop;
// nothing is GEMM-shaped (the contraction depth is |S| <= a few dims), so the
// bound for every kernel is memory bandwidth/latency or VALU issue, not MFMA.
//
// Floating point: the reference compares fl(sqrt(sum_k fl(fl(p_k - q_k)^2))) <= eps
// with separate multiplies and adds in subspace order (ClusteringCpu.cu:40-81).
// This file is compiled with -ffp-contract=off and the pragma below so that no
// multiply-add is fused, and the sqrt is replaced by the exact equivalent
// `sum <= s_star` (s_star = largest float whose sqrtf is <= eps).

#include <climits>
#include <cmath>
#include <cstring>


#include "inscy_device.h"
#include "inscy_internal.h"

#pragma clang fp contract(off)

namespace inscy {

namespace {


// ------------------------------------------------------------ discretisation
// get_cell_no (ScyTreeNode.cu:100-102): min((int)(x / (1/c)), c-1); the
// s-connection test of construct_s_connection (:34-49): x >= (c+1)*(1/c) - eps.
// cell of level t into the point's row, written 16 levels at a time
__device__ __forceinline__ void put_cell(uint8_t *__restrict__ rows, int rs, int p, int t, int d, int c, uint64_t &lo,
                                         uint64_t &hi) {
    if (!rows) return;
    const uint64_t v = (uint64_t) (uint8_t) c << (8 * (t & 7));
    if (t & 8)
        hi |= v;
    else
        lo |= v;
    if ((t & 15) != 15 && t != d - 1) return;
    *reinterpret_cast<uint4 *>(rows + (size_t) p * rs + (t & ~15)) =
        make_uint4((uint32_t) lo, (uint32_t) (lo >> 32), (uint32_t) hi, (uint32_t) (hi >> 32));
    lo = hi = 0;
}

__global__ void k_cell_rows(const uint8_t *__restrict__ cellC, int n, int d, const int *__restrict__ level,
                            uint8_t *__restrict__ rows, int rs) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    uint64_t lo = 0, hi = 0;
    for (int t = 0; t < d; ++t) put_cell(rows, rs, p, t, d, cellC[(size_t) level[t] * n + p], lo, hi);
}

__global__ void k_discretise(const float *__restrict__ X, int n, int d, int cells, float cs, int ecells,
                             float ecs, float eps, float *__restrict__ Xt, uint8_t *__restrict__ cellC,
                             uint16_t *__restrict__ cellE, uint8_t *__restrict__ rows, int rs,
                             uint64_t *__restrict__ nearw, int nw, int *__restrict__ bad) {
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    dmask_t nm = 0;
    bool out_of_range = false;
    uint64_t lo = 0, hi = 0;  // the cells of 16 dimensions
    for (int k = 0; k < d; ++k) {
        float x = X[(size_t) p * d + k];
        if (!(x >= 0.0f && x <= 1.0f)) out_of_range = true;
        x = fminf(fmaxf(x, 0.0f), 1.0f);  // keeps indices in range; the run is rejected via `bad`
        if (Xt) Xt[(size_t) k * n + p] = x;
        int c = min((int) __fdiv_rn(x, cs), cells - 1);
        int e = min((int) __fdiv_rn(x, ecs), ecells - 1);
        cellC[(size_t) k * n + p] = (uint8_t) c;
        cellE[(size_t) k * n + p] = (uint16_t) e;
        put_cell(rows, rs, p, k, d, c, lo, hi);
        float upper = __fmul_rn((float) (c + 1), cs);
        float bound = __fsub_rn(upper, eps);
        if (x >= bound) nm |= dbit(k);
    }
    // nw 64-bit words per point, dimension k at bit k % 64 of word k / 64
    nearw[(size_t) p * nw] = dlo(nm);
    if (nw > 1) nearw[(size_t) p * nw + 1] = dhi(nm);
    if (out_of_range) atomicOr(bad, 1);
}

// Occupancy of the ceil(1/eps)-grid per dimension; the host derives from it
// which dimensions of a subspace make the most selective grid index.
__global__ void k_hist1(const uint16_t *__restrict__ cellE, int n, int d, int ecells, int *__restrict__ hist) {
    size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t) n * d) return;
    int k = (int) (i / n);
    atomicAdd(&hist[(size_t) k * ecells + cellE[i]], 1);
}

// grid.y = dimension.  A few cells take all counts, so every block counts in LDS
// (n=3,001 d=9, 6 cells: 63 us with an atomic per value, 4.9 so).
constexpr int kHistItems = 8;
__global__ void k_histc(const uint8_t *__restrict__ cellC, int n, int cells, int *__restrict__ hist) {
    __shared__ int h[256];
    const int k = blockIdx.y;
    h[threadIdx.x] = 0;
    __syncthreads();
    for (int u = 0; u < kHistItems; ++u) {
        const int i = (blockIdx.x * kHistItems + u) * kBlock + threadIdx.x;
        if (i < n) atomicAdd(&h[cellC[(size_t) k * n + i]], 1);
    }
    __syncthreads();
    if (threadIdx.x < cells && h[threadIdx.x]) atomicAdd(&hist[(size_t) k * cells + threadIdx.x], h[threadIdx.x]);
}
static_assert(kBlock == 256, "one thread per possible cell");

// ------------------------------------------------------------ epsilon neighbourhood: subspace grid pass
// Candidate rule of get_possible_neighbors_from (ScyTreeNode.cu:896-946) on
// the ceil(1/eps)-grid: |cell_e(q) - cell_e(p)| <= 1 in every dimension of S;
// then the float distance in S (ClusteringCpu.cu:52-81).  Per subspace the
// points are counting-sorted by their cells in the j most selective
// dimensions of S (j <= 3), so the candidates of a query are 3^(j-1)
// contiguous ranges of the sorted order; the coordinates and cells of S are
// gathered into that order ([k][n]).  Queries run in the same sorted order and
// kLanesPerQuery lanes stride through each query's ranges, so the lanes of a
// wave read consecutive candidates and neighbouring queries share ranges.


__global__ void k_grid_keys(DevData D, SubspaceArg S, GridArg G, int *__restrict__ keys, int *__restrict__ rank,
                            int *__restrict__ hist) {
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= D.n) return;
    int key = 0;
    for (int a = 0; a < G.j; ++a) key = key * G.C + D.cellE[(size_t) S.dims[G.tI[a]] * D.n + p];
    keys[p] = key;
    rank[p] = atomicAdd(&hist[key], 1);
}

// Sorted order and the subspace's coordinates/cells gathered into it.
__global__ void k_grid_scatter(DevData D, SubspaceArg S, const int *__restrict__ keys, const int *__restrict__ rank,
                               const int *__restrict__ off, int *__restrict__ order, float *__restrict__ Ys,
                               uint16_t *__restrict__ Es) {
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= D.n) return;
    const int n = D.n;
    int pos = off[keys[p]] + rank[p];
    order[pos] = p;
    for (int t = 0; t < S.k; ++t) {
        int s = S.dims[t];
        Ys[(size_t) t * n + pos] = D.Xt[(size_t) s * n + p];
        Es[(size_t) t * n + pos] = D.cellE[(size_t) s * n + p];
    }
}


// |N_S(p)| of the points still uncounted (cnt == -1).  Counting stops once
// `cap` neighbours are found: every comparison made with a count is against a
// threshold <= cap, so min(|N_S(p)|, cap)-or-more decides them all.
__global__ __launch_bounds__(kBlock) void k_grid_count(int n, SubspaceArg S, GridArg G, const int *__restrict__ off,
                                                       const int *__restrict__ order, const float *__restrict__ Ys,
                                                       const uint16_t *__restrict__ Es, float s_star, int cap,
                                                       int *__restrict__ cnt) {
    constexpr int LPQ = kLanesPerQuery, QPB = kBlock / LPQ;
    extern __shared__ char smem[];
    float *sy = reinterpret_cast<float *>(smem);
    int *se = reinterpret_cast<int *>(smem + sizeof(float) * QPB * S.k);
    const int lq = threadIdx.x / LPQ, sub = threadIdx.x % LPQ;
    const int i = blockIdx.x * QPB + lq;
    int p = i < n ? order[i] : 0;
    const bool active = i < n && cnt[p] < 0;
    if (sub == 0 && active) stage_query(S, n, Ys, Es, i, sy + lq, se + lq, QPB);
    __syncthreads();
    int found = 0;
    if (active) {
        const float *qy = sy + lq;
        const int *qe = se + lq;
        const int gshift = (__lane_id() / LPQ) * LPQ;
        for_ranges(G, off, qe, QPB, [&](int a, int b) {
            for (int base = a; base < b && found < cap; base += LPQ) {
                int jj = base + sub;
                bool hit = jj < b && jj != i && is_neighbour(S, G, n, Ys, Es, qy, qe, QPB, jj, s_star);
                found += __popcll((__ballot(hit) >> gshift) & ((1ull << LPQ) - 1ull));
            }
        });
        if (sub == 0) cnt[p] = found;
    }
}

// dense flag per sorted position, union-find roots, zeroed component sizes
__global__ void k_dense_init(const int *__restrict__ order, int n, const int *__restrict__ cnt, int thr_dense,
                             uint8_t *__restrict__ dsorted, int *__restrict__ par, int *__restrict__ csize) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    // i: a sorted position for the dense flag, a point id for the rest
    dsorted[i] = cnt[order[i]] >= thr_dense ? 1 : 0;
    par[i] = cnt[i] >= thr_dense ? i : -1;
    csize[i] = 0;
}

// ------------------------------------------------------------ dense components
// Union-find over the dense-dense epsilon graph; hooking the larger root under
// the smaller keeps every root the smallest point id of its component, which
// is also the canonical cluster name.

// Components in the Afforest manner (Sutton, Ben-Nun, Bar-Noy, "Optimizing
// Parallel Graph Connectivity Computation via Subgraph Sampling", IPDPS 2018):
// (1) every dense point links to its first two dense neighbours, (2) roots are
// compressed, (3) the component holding most of a fixed sample of points is
// taken as the giant one, (4) only points outside it link to all their dense
// neighbours (both directions, so an edge between the giant component and the
// rest is still seen from the outside end).
__global__ __launch_bounds__(kBlock) void k_link_sample(int n, SubspaceArg S, GridArg G, const int *__restrict__ off,
                                                        const int *__restrict__ order, const float *__restrict__ Ys,
                                                        const uint16_t *__restrict__ Es,
                                                        const uint8_t *__restrict__ dsorted, float s_star,
                                                        int *__restrict__ par) {
    constexpr int LPQ = kLanesPerQuery, QPB = kBlock / LPQ;
    extern __shared__ char smem[];
    float *sy = reinterpret_cast<float *>(smem);
    int *se = reinterpret_cast<int *>(smem + sizeof(float) * QPB * S.k);
    const int lq = threadIdx.x / LPQ, sub = threadIdx.x % LPQ;
    const int i = blockIdx.x * QPB + lq;
    const bool active = i < n && dsorted[i];
    if (sub == 0 && active) stage_query(S, n, Ys, Es, i, sy + lq, se + lq, QPB);
    __syncthreads();
    if (!active) return;
    const float *qy = sy + lq;
    const int *qe = se + lq;
    const int p = order[i];
    const int gshift = (__lane_id() / LPQ) * LPQ;  // this query's lanes within the wave
    const unsigned long long below = (1ull << sub) - 1ull;
    int found = 0;
    for_ranges(G, off, qe, QPB, [&](int a, int b) {
        for (int base = a; base < b && found < 2; base += LPQ) {
            int jj = base + sub;
            bool hit = jj < b && jj != i && dsorted[jj] && is_neighbour(S, G, n, Ys, Es, qy, qe, QPB, jj, s_star);
            unsigned long long mine = (__ballot(hit) >> gshift) & ((1ull << LPQ) - 1ull);
            if (hit && __popcll(mine & below) < 2 - found) uf_union(par, p, order[jj]);
            found += min(__popcll(mine), 2 - found);
        }
    });
}

__global__ void k_uf_compress(int *__restrict__ par, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && par[i] >= 0) par[i] = uf_find(par, i);
}

// one block of 256: the most frequent root among 256 evenly spaced points
__global__ void k_giant(const int *__restrict__ par, int n, int *__restrict__ giant) {
    __shared__ int roots[256];
    __shared__ int best_c[256];
    __shared__ int best_r[256];
    const int t = threadIdx.x;
    int p = (int) (((long long) t * n) / 256);
    roots[t] = p < n ? par[p] : -1;
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
    if (t == 0) *giant = best_c[0] > 0 ? best_r[0] : -1;
}

__global__ __launch_bounds__(kBlock) void k_link_full(int n, SubspaceArg S, GridArg G, const int *__restrict__ off,
                                                      const int *__restrict__ order, const float *__restrict__ Ys,
                                                      const uint16_t *__restrict__ Es,
                                                      const uint8_t *__restrict__ dsorted, float s_star,
                                                      const int *__restrict__ giant, int *__restrict__ par) {
    constexpr int LPQ = kLanesPerQuery, QPB = kBlock / LPQ;
    extern __shared__ char smem[];
    float *sy = reinterpret_cast<float *>(smem);
    int *se = reinterpret_cast<int *>(smem + sizeof(float) * QPB * S.k);
    const int lq = threadIdx.x / LPQ, sub = threadIdx.x % LPQ;
    const int i = blockIdx.x * QPB + lq;
    bool active = i < n && dsorted[i];
    int p = active ? order[i] : 0;
    if (active && par[p] == *giant) active = false;
    if (sub == 0 && active) stage_query(S, n, Ys, Es, i, sy + lq, se + lq, QPB);
    __syncthreads();
    if (!active) return;
    const float *qy = sy + lq;
    const int *qe = se + lq;
    int rp = uf_find(par, p);
    for_ranges(G, off, qe, QPB, [&](int a, int b) {
        for (int jj = a + sub; jj < b; jj += LPQ) {
            if (jj == i || !dsorted[jj] || !is_neighbour(S, G, n, Ys, Es, qy, qe, QPB, jj, s_star)) continue;
            int q = order[jj];
            if (uf_find(par, q) == rp) continue;
            uf_union(par, p, q);
            rp = uf_find(par, p);
        }
    });
}

__global__ void k_uf_flatten(int *__restrict__ par, int n, int *__restrict__ comp, int *__restrict__ csize) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    int c = -1;
    if (i < n && par[i] >= 0) c = uf_find(par, i);
    wave_add_by_key(csize, c, c >= 0);
    if (i < n) comp[i] = c;
}

// Canonical labels of a chunk of result subspaces (grid.y = row): clusters
// are numbered by their smallest point id, which is the component root.
// Pass 1 flags the kept roots, an exclusive scan over the whole chunk numbers
// them, pass 2 writes every point's number relative to its row's first root.
__global__ void k_emit_roots(const EmitRow *__restrict__ rows, int n, int *__restrict__ flags) {
    const EmitRow R = rows[blockIdx.y];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (i == 0 && blockIdx.y == 0) flags[(size_t) gridDim.y * n] = 0;  // the scan's last entry is the total
    flags[(size_t) blockIdx.y * n + i] = (R.comp[i] == i && R.inres[i]) ? 1 : 0;
}

// T = int: the label; T = uint8_t / uint16_t: the label + 1 (0 for noise), for
// rows whose labels fit (the host reads them back at a quarter or half the bytes)
template <class T>
__global__ void k_emit_labels(const EmitRow *__restrict__ rows, int n, const int *__restrict__ idx,
                              T *__restrict__ labels, int *__restrict__ counts) {
    const EmitRow R = rows[blockIdx.y];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const size_t row = (size_t) blockIdx.y * n;
    if (i == 0) counts[blockIdx.y] = idx[row + n] - idx[row];
    const int c = R.comp[i];
    const int v = (c >= 0 && R.inres[c]) ? idx[row + c] - idx[row] : -1;
    labels[row + i] = (T) (sizeof(T) == sizeof(int) ? v : v + 1);
}

template <class T>
__global__ void k_fill(T *p, T v, size_t count) {
    fill_span(p, v, count);
}

struct FillArgs {
    FillMany f;
    int blk[FillMany::kMost + 1];  // first block of each array
};
constexpr int kFillVecs = 8;  // 16-byte stores per thread
__global__ __launch_bounds__(kBlock) void k_fill_many(FillArgs a) {
    int s = 0;
    while (s + 1 < a.f.n && (int) blockIdx.x >= a.blk[s + 1]) ++s;
    const uint32_t v = a.f.v[s];
    const size_t words = a.f.words[s], nvec = words / 4;
    uint4 *q = reinterpret_cast<uint4 *>(a.f.p[s]);
    const size_t step = (size_t) (a.blk[s + 1] - a.blk[s]) * kBlock;
    const size_t t0 = (size_t) (blockIdx.x - a.blk[s]) * kBlock + threadIdx.x;
    for (size_t j = t0; j < nvec; j += step) q[j] = make_uint4(v, v, v, v);
    if (t0 < words - 4 * nvec) a.f.p[s][4 * nvec + t0] = v;
}

__global__ void k_gather(const int *__restrict__ src, const int *__restrict__ idx, int count, int *__restrict__ out) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) out[i] = src[idx[i]];
}

__global__ void k_iota(int *__restrict__ p, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = i;
}

__global__ void k_rank_keys(const uint16_t *__restrict__ cellE, int n, int dim, const int *__restrict__ perm,
                            uint16_t *__restrict__ keys) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) keys[i] = cellE[(size_t) dim * n + perm[i]];
}

}  // namespace

// ------------------------------------------------------------ launchers
float sqrt_threshold(float eps) {
    // bisection on the ordered bit patterns of non-negative floats
    uint32_t lo = 0, hi = 0x7f800000u;  // [0, +inf)
    auto sq = [](uint32_t b) {
        float f;
        std::memcpy(&f, &b, 4);
        return sqrtf(f);
    };
    if (!(sq(lo) <= eps)) return -1.0f;
    while (hi - lo > 1) {
        uint32_t mid = lo + (hi - lo) / 2;
        if (sq(mid) <= eps)
            lo = mid;
        else
            hi = mid;
    }
    float f;
    std::memcpy(&f, &lo, 4);
    return f;
}

#define LAUNCH(kernel, grid, block, lds, st, ...) hipLaunchKernelGGL(kernel, grid, block, lds, st, __VA_ARGS__)

hipError_t launch_cell_rows(const uint8_t *cellC, int n, int d, const int *level, uint8_t *rows, hipStream_t st) {
    LAUNCH(k_cell_rows, dim3(blocks_for(n)), dim3(kBlock), 0, st, cellC, n, d, level, rows, cell_row_bytes(d));
    return hipGetLastError();
}

hipError_t launch_discretise(const float *X, int n, int d, int cells, float eps, float *Xt, uint8_t *cellC,
                             uint16_t *cellE, uint8_t *rows, uint64_t *nearw, int nw, int *bad, hipStream_t st) {
    int ecells = (int) ceil(1.0 / (double) eps);
    float cs = 1.0f / (float) cells;
    float ecs = 1.0f / (float) ecells;
    LAUNCH(k_discretise, dim3(blocks_for(n)), dim3(kBlock), 0, st, X, n, d, cells, cs, ecells, ecs, eps, Xt, cellC,
           cellE, rows, cell_row_bytes(d), nearw, nw, bad);
    return hipGetLastError();
}

hipError_t launch_hist1(const uint16_t *cellE, int n, int d, int ecells, int *hist, hipStream_t st) {
    size_t nd = (size_t) n * d;
    LAUNCH(k_hist1, dim3(blocks_for(nd)), dim3(kBlock), 0, st, cellE, n, d, ecells, hist);
    return hipGetLastError();
}

hipError_t launch_histc(const uint8_t *cellC, int n, int d, int cells, int *hist, hipStream_t st) {
    LAUNCH(k_fill<int>, dim3(fill_blocks((size_t) d * cells, sizeof(int))), dim3(kBlock), 0, st, hist, 0, (size_t) d * cells);
    LAUNCH(k_histc, dim3((n + kBlock * kHistItems - 1) / (kBlock * kHistItems), d), dim3(kBlock), 0, st, cellC, n,
           cells, hist);
    return hipGetLastError();
}


static hipError_t build_grid(const DevData &D, const SubspaceArg &S, const GridArg &G, const GridBuffers &B,
                             hipStream_t st) {
    const int n = D.n;
    int ncell = 1;
    for (int a = 0; a < G.j; ++a) ncell *= G.C;
    LAUNCH(k_fill<int>, dim3(fill_blocks((size_t) ncell + 1, sizeof(int))), dim3(kBlock), 0, st, B.hist, 0, (size_t) ncell + 1);
    LAUNCH(k_grid_keys, dim3(blocks_for(n)), dim3(kBlock), 0, st, D, S, G, B.keys, B.rank, B.hist);
    hipError_t e = launch_exclusive_sum(B.scan_temp, B.scan_bytes, B.hist, B.off, ncell + 1, st);
    if (e != hipSuccess) return e;
    LAUNCH(k_grid_scatter, dim3(blocks_for(n)), dim3(kBlock), 0, st, D, S, B.keys, B.rank, B.off, B.order, B.Ys, B.Es);
    return hipGetLastError();
}

static unsigned query_blocks(int n) {
    return (unsigned) ((n + kBlock / kLanesPerQuery - 1) / (kBlock / kLanesPerQuery));
}

static size_t query_lds(const SubspaceArg &S) { return (sizeof(float) + sizeof(int)) * (kBlock / kLanesPerQuery) * S.k; }

hipError_t launch_subspace_counts(const DevData &D, const SubspaceArg &S, const GridArg &G, float s_star, int cap,
                                  const GridBuffers &B, int *cnt, hipStream_t st) {
    hipError_t e = build_grid(D, S, G, B, st);
    if (e != hipSuccess) return e;
    LAUNCH(k_grid_count, dim3(query_blocks(D.n)), dim3(kBlock), query_lds(S), st, D.n, S, G, B.off, B.order, B.Ys,
           B.Es, s_star, cap, cnt);
    return hipGetLastError();
}

hipError_t launch_subspace_components(const DevData &D, const SubspaceArg &S, const GridArg &G, float s_star,
                                      int cap, int thr_dense, const GridBuffers &B, int *cnt, int *comp,
                                      int *csize, hipStream_t st) {
    hipError_t e = build_grid(D, S, G, B, st);
    if (e != hipSuccess) return e;
    const int n = D.n;
    LAUNCH(k_grid_count, dim3(query_blocks(n)), dim3(kBlock), query_lds(S), st, n, S, G, B.off, B.order, B.Ys, B.Es,
           s_star, cap, cnt);
    LAUNCH(k_dense_init, dim3(blocks_for(n)), dim3(kBlock), 0, st, B.order, n, cnt, thr_dense, B.dsorted, B.par,
           csize);
    LAUNCH(k_link_sample, dim3(query_blocks(n)), dim3(kBlock), query_lds(S), st, n, S, G, B.off, B.order, B.Ys, B.Es,
           B.dsorted, s_star, B.par);
    LAUNCH(k_uf_compress, dim3(blocks_for(n)), dim3(kBlock), 0, st, B.par, n);
    LAUNCH(k_giant, dim3(1), dim3(256), 0, st, B.par, n, B.giant);
    LAUNCH(k_link_full, dim3(query_blocks(n)), dim3(kBlock), query_lds(S), st, n, S, G, B.off, B.order, B.Ys, B.Es,
           B.dsorted, s_star, B.giant, B.par);
    LAUNCH(k_uf_flatten, dim3(blocks_for(n)), dim3(kBlock), 0, st, B.par, n, comp, csize);
    return hipGetLastError();
}

hipError_t launch_emit(const EmitRow *rows, int r, int n, int *flags, int *idx, void *labels, int width, int *counts,
                       void *scan_temp, size_t scan_bytes, hipStream_t st) {
    if (r <= 0) return hipSuccess;
    const size_t items = (size_t) r * n + 1;
    LAUNCH(k_emit_roots, dim3(blocks_for(n), r), dim3(kBlock), 0, st, rows, n, flags);
    hipError_t e = launch_exclusive_sum(scan_temp, scan_bytes, flags, idx, (int) items, st);
    if (e != hipSuccess) return e;
    if (width == 1)
        LAUNCH(k_emit_labels<uint8_t>, dim3(blocks_for(n), r), dim3(kBlock), 0, st, rows, n, idx,
               static_cast<uint8_t *>(labels), counts);
    else if (width == 2)
        LAUNCH(k_emit_labels<uint16_t>, dim3(blocks_for(n), r), dim3(kBlock), 0, st, rows, n, idx,
               static_cast<uint16_t *>(labels), counts);
    else
        LAUNCH(k_emit_labels<int>, dim3(blocks_for(n), r), dim3(kBlock), 0, st, rows, n, idx,
               static_cast<int *>(labels), counts);
    return hipGetLastError();
}

hipError_t launch_fill_u64(uint64_t *p, uint64_t v, size_t count, hipStream_t st) {
    if (!count) return hipSuccess;
    LAUNCH(k_fill<uint64_t>, dim3(fill_blocks(count, sizeof(uint64_t))), dim3(kBlock), 0, st, p, v, count);
    return hipGetLastError();
}

hipError_t launch_fill_i32(int *p, int v, size_t count, hipStream_t st) {
    if (!count) return hipSuccess;
    LAUNCH(k_fill<int>, dim3(fill_blocks(count, sizeof(int))), dim3(kBlock), 0, st, p, v, count);
    return hipGetLastError();
}

hipError_t launch_fill_many(const FillMany &f, hipStream_t st) {
    if (f.n <= 0) return hipSuccess;
    FillArgs a{f, {}};
    a.blk[0] = 0;
    for (int s = 0; s < f.n; ++s) {
        const size_t b = (f.words[s] / 4 + kBlock * kFillVecs - 1) / (kBlock * kFillVecs);
        a.blk[s + 1] = a.blk[s] + (int) std::max<size_t>(1, std::min<size_t>(b, 4096));
    }
    LAUNCH(k_fill_many, dim3(a.blk[f.n]), dim3(kBlock), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_gather(const int *src, const int *idx, int count, int *out, hipStream_t st) {
    if (count <= 0) return hipSuccess;
    LAUNCH(k_gather, dim3(blocks_for(count)), dim3(kBlock), 0, st, src, idx, count, out);
    return hipGetLastError();
}

size_t rank_order_temp_bytes(int n) { return sort_temp_bytes(n); }

// Least-significant dimension first, one stable radix sort per dimension (one
// or two 8-bit digit passes for cells below ecells), starting from ascending
// ids: the result is sorted by the cells in `level` order with ties by id.
hipError_t launch_rank_order(const uint16_t *cellE, int n, int d, int ecells, const int *level, int *perm, int *tmp,
                             uint16_t *keys, uint16_t *keys2, void *temp, size_t temp_bytes, hipStream_t st) {
    LAUNCH(k_iota, dim3(blocks_for(n)), dim3(kBlock), 0, st, perm, n);
    int bits = 1;
    while (bits < 16 && (1 << bits) < ecells) ++bits;
    const bool two = bits > 8;
    int *a = perm, *b = tmp;
    for (int t = d - 1; t >= 0; --t) {
        LAUNCH(k_rank_keys, dim3(blocks_for(n)), dim3(kBlock), 0, st, cellE, n, level[t], a, keys);
        // two passes: keys -> keys2 -> keys and a -> b -> a; one pass: keys -> keys2 and a -> b
        hipError_t e = launch_sort_pairs_u16(keys, keys2, two ? keys : keys2, a, b, two ? a : b, n, bits, temp,
                                             temp_bytes, st);
        if (e != hipSuccess) return e;
        if (!two) {
            int *x = a;
            a = b;
            b = x;
        }
    }
    if (a != perm) {
        hipError_t e = hipMemcpyAsync(perm, a, (size_t) n * sizeof(int), hipMemcpyDeviceToDevice, st);
        if (e != hipSuccess) return e;
    }
    return hipGetLastError();
}

}  // namespace inscy
