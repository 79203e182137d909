// k_wcc.hip -- weakly connected components by min-label propagation.
//
// Reference: wcc.cu:140-485.  Per round the reference joins the delta
// Δ(n, l) with the symmetric edge relation, merges the result into
// cc(node, label), keeps the minimum label per node (unique_by_key after a
// sorted merge) and takes Δ' = cc' \ cc.  The same relation is computed here
// on dense node ids (the sorted distinct keys of the symmetric edge set):
//   L[v]      current label of node v (a dense id; dense order == id order,
//             so min over dense ids == min over the original ids)
//   frontier  (v, l) pairs of Δ; l is the label v had when it entered Δ, so
//             sources read a snapshot (Jacobi), exactly as the reference's
//             join reads Δ's value column
//   relax     for every edge (v, m) of a frontier node: atomicMin(L[m], l);
//             a node whose label dropped is appended once per round
//             (mark[m] == round), giving Δ' = {(m, L'(m)) : L'(m) < L(m)}
// Edge traversal is load balanced: degree counts -> scan -> one thread per
// edge, its node found from the tile's node starts set as bits in LDS.
//
// Two other forms of the same round (same labels, same Δ'):
//   round one  every node is in Δ with its own id as label, so L'(m) is the
//              least of m and its neighbours; neighbour lists are sorted
//              (the index keeps each key's rows in value order), so that is
//              min(m, first neighbour): one read per node instead of per edge
//   pull       L'(m) = min(L(m), min over ALL neighbours v of L(v)).  Equal to
//              the push round because a neighbour v outside Δ has already
//              pushed its current label: v's label last changed in a round
//              after which v was in Δ, and the next round lowered m to it
//              (round one has every node in Δ).  One thread per edge again,
//              but reading labels instead of taking atomics: a segmented
//              minimum over the wave's lanes of one node, then one atomic per
//              node and wave into a copy Ln of L; Δ' = {m : Ln(m) < L(m)}.
#include "dlg_internal.h"

#include <algorithm>
#include <chrono>
#include <deque>
#include <memory>

namespace dlg {

__global__ void wcc_init_k(u32 *L, u32 *fnode, u32 *flabel, u32 *mark, u64 V) {
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    u64 stride = (u64)gridDim.x * blockDim.x;
    for (; i < V; i += stride) {
        L[i] = (u32)i;
        fnode[i] = (u32)i;
        flabel[i] = (u32)i;
        mark[i] = 0;
    }
}

__global__ void wcc_degree_k(const u32 *fnode, u64 nf, const u32 *gstart, u32 *cnt, u32 *pstart) {
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    u64 stride = (u64)gridDim.x * blockDim.x;
    for (; i < nf; i += stride) {
        u32 v = fnode[i];
        u32 s = gstart[v];
        cnt[i] = gstart[v + 1] - s;
        pstart[i] = s;
    }
}

// Appends of a block's tile with ONE counter atomic per block: an atomic per
// wave on one address serialises over the whole grid (~70k waves for a
// round that lowers 4.6M nodes).  Each thread offers I items; the slots
// follow (item, wave, lane) order.  s_cnt: I * T / WAVE + 1 u32 of LDS, at
// most 65.  Every thread of the block must call it.
template <int T, int I>
__device__ __forceinline__ void block_append(const bool (&app)[I], u32 *count, u32 *s_cnt, u32 (&slot)[I]) {
    constexpr int W = T / WAVE, K = I * W;
    static_assert(K <= WAVE, "one wave scans the per-wave counts");
    const int wave = threadIdx.x / WAVE, lane = threadIdx.x & (WAVE - 1);
    u64 bm[I];
#pragma unroll
    for (int r = 0; r < I; r++) {
        bm[r] = __ballot(app[r]);
        if (lane == 0) s_cnt[r * W + wave] = (u32)__popcll(bm[r]);
    }
    __syncthreads();
    if (wave == 0) {
        const u32 c = lane < K ? s_cnt[lane] : 0u;
        u32 tot = 0;
        const u32 ex = wave_excl_scan32(c, &tot);
        u32 b = 0;
        if (lane == 0 && tot) b = atomicAdd(count, tot);
        b = __shfl(b, 0, WAVE);
        if (lane < K) s_cnt[lane] = b + ex;
    }
    __syncthreads();
    const u64 lt = lanemask_lt();
#pragma unroll
    for (int r = 0; r < I; r++) slot[r] = s_cnt[r * W + wave] + (u32)__popcll(bm[r] & lt);
    __syncthreads();   // s_cnt may be reused
}

// The owners of a tile's TS_TILE positions (edges, or join rows) base ..
// base + TS_TILE - 1 under offsets that rise strictly (every node has an
// edge): offs[lo] <= base and nodes lo+1 .. hi-1 start inside the tile.  Their
// starts are set as bits in LDS; the owner of tile position p is lo plus the
// starts at or before p -- what a binary search of offs gives, without global
// loads per position.
constexpr int TS_TILE = 2048, TS_WORDS = TS_TILE / 32;
static_assert(TS_WORDS == WAVE, "one wave scans the start words");
struct TileStarts {
    u32 bits[TS_WORDS];     // bit p: a node starts at base + p
    u32 before[TS_WORDS];   // starts in the words before
};

// Before the caller's barrier that publishes lo and hi.
__device__ __forceinline__ void tile_starts_clear(TileStarts &ts) {
    if (threadIdx.x < TS_WORDS) ts.bits[threadIdx.x] = 0u;
}

// Every thread of the block calls it (two barriers).
template <int T, typename O>
__device__ __forceinline__ void tile_starts_set(TileStarts &ts, const O *offs, u64 lo, u64 hi, u64 base) {
    for (u64 j = lo + 1 + threadIdx.x; j < hi; j += T) {   // base < offs[j] < base + TS_TILE
        const u32 p = (u32)((u64)offs[j] - base);
        atomicOr(&ts.bits[p >> 5], 1u << (p & 31u));
    }
    __syncthreads();
    if (threadIdx.x < WAVE) {
        u32 tot;
        ts.before[threadIdx.x] = wave_excl_scan32((u32)__popc(ts.bits[threadIdx.x]), &tot);
    }
    __syncthreads();
}

// Owner of tile position p (< TS_TILE), relative to lo.
__device__ __forceinline__ u32 tile_owner(const TileStarts &ts, u32 p) {
    return ts.before[p >> 5] + (u32)__popc(ts.bits[p >> 5] & (0xffffffffu >> (31u - (p & 31u))));
}

constexpr int WR_T = 256, WR_I = 8, WR_TILE = WR_T * WR_I;
static_assert(WR_TILE == TS_TILE, "relax tiles");

__global__ __launch_bounds__(WR_T) void wcc_relax_k(const u32 *flabel, u64 nf, const u32 *pstart,
                                                    const u64 *offs, u64 total, const u32 *nbr,
                                                    u32 *L, u32 *mark, u32 round, u32 *next_node,
                                                    u32 *next_count) {
    __shared__ u64 s_lo, s_hi;
    __shared__ u32 s_cnt[WR_I * WR_T / WAVE + 1];
    __shared__ TileStarts ts;
    const u64 base = (u64)blockIdx.x * WR_TILE;
    tile_starts_clear(ts);
    if (threadIdx.x < WAVE) {   // the first wave finds the tile's frontier nodes
        const u64 last = (base + WR_TILE < total ? base + WR_TILE : total) - 1;
        const u64 lo = wave_upper_bound(offs, 0, nf, base) - 1;
        const u64 hi = wave_upper_bound(offs, lo, nf, last);
        if (threadIdx.x == 0) {
            s_lo = lo;
            s_hi = hi;
        }
    }
    __syncthreads();
    const u64 lo = s_lo, hi = s_hi;
    tile_starts_set<WR_T>(ts, offs, lo, hi, base);   // frontier nodes have edges: offsets rise strictly
    bool app[WR_I];
    u32 m[WR_I], slot[WR_I];
#pragma unroll
    for (int r = 0; r < WR_I; r++) {
        u64 o = base + (u64)r * WR_T + threadIdx.x;
        app[r] = false;
        m[r] = 0;
        if (o < total) {
            const u64 i = lo + tile_owner(ts, (u32)(r * WR_T) + threadIdx.x);
            m[r] = nbr[(u64)pstart[i] + (o - offs[i])];
            u32 l = flabel[i];
            if (L[m[r]] > l) {
                u32 old = atomicMin(&L[m[r]], l);
                if (old > l) app[r] = atomicExch(&mark[m[r]], round) != round;
            }
        }
    }
    block_append<WR_T, WR_I>(app, next_count, s_cnt, slot);
#pragma unroll
    for (int r = 0; r < WR_I; r++)
        if (app[r]) next_node[slot[r]] = m[r];
}

constexpr int WA_T = 256, WA_I = 16, WA_TILE = WA_T * WA_I;   // node-parallel kernels: one tile per block

// Round one: L(m) = min(m, first neighbour of m); lowered nodes appended with
// their label.  Every node has a neighbour (the nodes are the edge keys).
__global__ __launch_bounds__(WA_T) void wcc_first_k(const u32 *gstart, const u32 *nbr, u64 V, u32 *L,
                                                    u32 *next_node, u32 *next_label, u32 *count) {
    __shared__ u32 s_cnt[WA_I * WA_T / WAVE + 1];
    const u64 base = (u64)blockIdx.x * WA_TILE;
    bool app[WA_I];
    u32 l[WA_I], slot[WA_I];
#pragma unroll
    for (int r = 0; r < WA_I; r++) {
        const u64 i = base + (u64)r * WA_T + threadIdx.x;
        app[r] = false;
        l[r] = 0;
        if (i < V) {
            const u32 f = nbr[gstart[i]];
            app[r] = f < (u32)i;
            l[r] = app[r] ? f : (u32)i;
            if (app[r]) L[i] = l[r];
        }
    }
    block_append<WA_T, WA_I>(app, count, s_cnt, slot);
#pragma unroll
    for (int r = 0; r < WA_I; r++)
        if (app[r]) {
            next_node[slot[r]] = (u32)(base + (u64)r * WA_T + threadIdx.x);
            next_label[slot[r]] = l[r];
        }
}

// Pull round over all ne edges (CSR gstart/nbr): Ln(m) = min(Ln(m), L(v)) for
// every edge (m, v), with Ln == L on entry.  A thread takes 8 edges in a row, whose
// nodes come from the tile's node starts (TileStarts), and gives every node's least
// to the tile's minima in LDS; only a tile's first and last node can have edges in
// other tiles.  Nodes with label 0 read no labels: nothing is below it, and the
// component of the least id is most of a graph that is worth a pull.
// Bound by the label reads, one L2 line a lane.  With a segmented minimum over each
// wave (12 LDS shuffles for 64 edges) and every label read, R-MAT-23's 2.6e8 edges
// took 1.85 ms a round; they take 0.78.
constexpr int WP_T = 256, WP_I = 8, WP_TILE = WP_T * WP_I;
static_assert(WP_TILE == TS_TILE, "pull tiles");

__global__ __launch_bounds__(WP_T) void wcc_pull_k(const u32 *gstart, u64 V, u64 ne, const u32 *nbr,
                                                   const u32 *L, u32 *Ln) {
    __shared__ u64 s_lo, s_hi;
    __shared__ TileStarts ts;
    __shared__ u32 s_min[WP_TILE + 1];
    const u64 base = (u64)blockIdx.x * WP_TILE;
    const u32 p0 = threadIdx.x * WP_I, have = base + p0 < ne ? (u32)min(ne - base - p0, (u64)WP_I) : 0u;
    u32 v[WP_I];
    if (have == WP_I) {
#pragma unroll
        for (int j = 0; j < WP_I; j += 4) {   // nbr is a block of its own and p0 a multiple of 8: aligned
            const uint4 q = *(const uint4 *)(nbr + base + p0 + j);
            v[j] = q.x; v[j + 1] = q.y; v[j + 2] = q.z; v[j + 3] = q.w;
        }
    } else {
#pragma unroll
        for (int j = 0; j < WP_I; j++) v[j] = (u32)j < have ? nbr[base + p0 + j] : 0u;
    }
    tile_starts_clear(ts);
    if (threadIdx.x < WAVE) {   // the first wave finds the tile's nodes
        const u64 last = (base + WP_TILE < ne ? base + WP_TILE : ne) - 1;
        const u64 lo = wave_upper_bound(gstart, 0, V, base) - 1;
        const u64 hi = wave_upper_bound(gstart, lo, V, last);
        if (threadIdx.x == 0) {
            s_lo = lo;
            s_hi = hi;
        }
    }
    __syncthreads();
    const u64 lo = s_lo;
    const u32 nodes = (u32)(s_hi - lo);   // at most one starting at every position, and one before
    for (u32 i = threadIdx.x; i < nodes; i += WP_T) s_min[i] = L[lo + i];
    tile_starts_set<WP_T>(ts, gstart, lo, lo + nodes, base);
    const u32 starts = (ts.bits[p0 >> 5] >> (p0 & 31u)) & 0xffu;
    u32 own[WP_I];
    bool need[WP_I];
    own[0] = tile_owner(ts, p0);
#pragma unroll
    for (int j = 0; j < WP_I; j++) {
        if (j) own[j] = own[j - 1] + ((starts >> j) & 1u);
        need[j] = (u32)j < have && s_min[own[j]] != 0u;   // past the end: the last node, in range
    }
    __syncthreads();   // read before they are lowered
    u32 val[WP_I];
#pragma unroll
    for (int j = 0; j < WP_I; j++) val[j] = need[j] ? L[v[j]] : 0xffffffffu;
    u32 cur = val[0];
    const u32 first = (u32)__builtin_amdgcn_readfirstlane((int)own[0]);
    if (__all(own[WP_I - 1] == first)) {   // a hub's edges, the whole wave's
#pragma unroll
        for (int j = 1; j < WP_I; j++) cur = min(cur, val[j]);
#pragma unroll
        for (int d = WAVE / 2; d > 0; d >>= 1) cur = min(cur, (u32)__shfl_xor((int)cur, d, WAVE));
        if ((threadIdx.x & (WAVE - 1)) == 0 && cur != 0xffffffffu) atomicMin(&s_min[first], cur);
    } else {
#pragma unroll
        for (int j = 1; j < WP_I; j++) {
            if (own[j] != own[j - 1]) {
                if (cur != 0xffffffffu) atomicMin(&s_min[own[j - 1]], cur);
                cur = 0xffffffffu;
            }
            cur = min(cur, val[j]);
        }
        if (cur != 0xffffffffu) atomicMin(&s_min[own[WP_I - 1]], cur);
    }
    __syncthreads();
    for (u32 i = threadIdx.x; i < nodes; i += WP_T) {
        const u32 m = s_min[i];
        if (m >= L[lo + i]) continue;
        if (i == 0 || i + 1 == nodes) atomicMin(&Ln[lo + i], m);
        else Ln[lo + i] = m;
    }
}

// Δ' of a pull round: nodes whose label dropped, appended with the new label;
// L takes the new labels, so L == Ln again afterwards.
__global__ __launch_bounds__(WA_T) void wcc_changed_k(u32 *L, const u32 *Ln, u64 V, u32 *next_node,
                                                      u32 *next_label, u32 *count) {
    __shared__ u32 s_cnt[WA_I * WA_T / WAVE + 1];
    const u64 base = (u64)blockIdx.x * WA_TILE;
    bool app[WA_I];
    u32 l[WA_I], slot[WA_I];
#pragma unroll
    for (int r = 0; r < WA_I; r++) {
        const u64 i = base + (u64)r * WA_T + threadIdx.x;
        app[r] = false;
        l[r] = 0;
        if (i < V) {
            l[r] = Ln[i];
            app[r] = l[r] < L[i];
            if (app[r]) L[i] = l[r];
        }
    }
    block_append<WA_T, WA_I>(app, count, s_cnt, slot);
#pragma unroll
    for (int r = 0; r < WA_I; r++)
        if (app[r]) {
            next_node[slot[r]] = (u32)(base + (u64)r * WA_T + threadIdx.x);
            next_label[slot[r]] = l[r];
        }
}

__global__ void wcc_gather_k(const u32 *node, u64 n, const u32 *L, u32 *label) {
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    u64 stride = (u64)gridDim.x * blockDim.x;
    for (; i < n; i += stride) label[i] = L[node[i]];
}

// Nodes per label.  A giant component's label covers most of every tile, and
// one atomic per wave on its counter would serialise over the grid: the
// tile's first label is counted in registers and added once per block; the
// other labels go through per-wave grouping.
__global__ __launch_bounds__(WA_T) void wcc_comp_count_k(const u32 *L, u64 V, u32 *ccount) {
    __shared__ u32 s_part[WA_T / WAVE];
    const u64 base = (u64)blockIdx.x * WA_TILE;
    const u32 hot = L[base];
    u32 mine = 0;
#pragma unroll
    for (int r = 0; r < WA_I; r++) {
        const u64 i = base + (u64)r * WA_T + threadIdx.x;
        const bool valid = i < V;
        const u32 k = valid ? L[i] : 0u;
        mine += (valid && k == hot) ? 1u : 0u;
        wave_count_by_key(ccount, k, valid && k != hot);
    }
#pragma unroll
    for (int d = WAVE / 2; d > 0; d >>= 1) mine += (u32)__shfl_xor((int)mine, d, WAVE);
    if ((threadIdx.x & (WAVE - 1)) == 0) s_part[threadIdx.x / WAVE] = mine;
    __syncthreads();
    if (threadIdx.x == 0) {
        u32 s = 0;
        for (int w = 0; w < WA_T / WAVE; w++) s += s_part[w];
        atomicAdd(&ccount[hot], s);
    }
}

// flags[v] = ccount[v] > 0; largest via atomicMax.
__global__ void wcc_comp_flags_k(const u32 *ccount, u64 V, u32 *flags, u32 *largest) {
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    u64 stride = (u64)gridDim.x * blockDim.x;
    u32 mx = 0;
    for (; i < V; i += stride) {
        u32 c = ccount[i];
        flags[i] = c > 0 ? 1u : 0u;
        mx = max(mx, c);
    }
#pragma unroll
    for (int d = WAVE / 2; d > 0; d >>= 1) mx = max(mx, (u32)__shfl_xor((int)mx, d, WAVE));
    if ((threadIdx.x & (WAVE - 1)) == 0 && mx) atomicMax(largest, mx);
}

// Output tuples (node key, 0) for every label in use, in node order.
__global__ void wcc_emit_k(const u32 *flags, const u64 *offs, u64 V, const u64 *rows,
                           const u32 *gstart, u64 *out) {
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    u64 stride = (u64)gridDim.x * blockDim.x;
    for (; i < V; i += stride)
        if (flags[i]) out[offs[i]] = tmake(tkey(rows[gstart[i]]), 0x80000000u);
}

static u64 read_counter(dlg_ctx *ctx, WccState &s) {
    u32 h = 0;
    ctx->read_words(s.counter.p, 1, &h);
    return h;
}

u64 wcc_first_round(dlg_ctx *ctx, WccState &s, const Index &ix, const u32 *nbr) {
    const u64 V = s.V;
    if (V == 0) return 0;
    fill_u32(ctx, s.counter.p, 1, 0u);
    // 4 B start + 4 B first neighbour per node; lowered nodes: 4 B label + 8 B appended
    DLG_LAUNCH(ctx, DLG_K_WCC_RELAX, 8.0 * V, wcc_first_k, grid_for(V, WA_TILE), WA_T, 0,
               (const u32 *)ix.gstart.p, nbr, V, s.L.p, s.fnode.p, s.flabel.p, s.counter.p);
    return read_counter(ctx, s);
}

static u64 wcc_pull_round(dlg_ctx *ctx, WccState &s, const Index &ix, const u32 *nbr) {
    const u64 V = s.V, ne = ix.n;
    s.Ln.ensure(V);
    HIPCHK(hipMemcpyAsync(s.Ln.p, s.L.p, V * 4, hipMemcpyDeviceToDevice, ctx->stream));
    fill_u32(ctx, s.counter.p, 1, 0u);
    if (ne)
        // 4 B neighbour id + 4 B label read per edge; per node 4 B start and 4 B Ln
        DLG_LAUNCH(ctx, DLG_K_WCC_RELAX, 8.0 * ne + 8.0 * V, wcc_pull_k, grid_for(ne, WP_TILE), WP_T, 0,
                   (const u32 *)ix.gstart.p, V, ne, nbr, (const u32 *)s.L.p, s.Ln.p);
    DLG_LAUNCH(ctx, DLG_K_WCC_RELAX, 8.0 * V, wcc_changed_k, grid_for(V, WA_TILE), WA_T, 0, s.L.p,
               (const u32 *)s.Ln.p, V, s.nnode.p, s.flabel.p, s.counter.p);
    s.fnode.swap(s.nnode);
    return read_counter(ctx, s);
}

// One round.  Returns |Δ'| (the new frontier size); the frontier is replaced.
u64 wcc_round(dlg_ctx *ctx, WccState &s, const Index &ix, const u32 *nbr, u64 nf, u32 round, int form) {
    if (form == WCC_PULL) return wcc_pull_round(ctx, s, ix, nbr);
    s.cnt.ensure(nf);
    s.pstart.ensure(nf);
    s.offs.ensure(nf + 1);
    DLG_LAUNCH(ctx, DLG_K_WCC_RELAX, 16.0 * nf, wcc_degree_k, sgrid(ctx, nf), ctx->block_size, 0,
               (const u32 *)s.fnode.p, nf, (const u32 *)ix.gstart.p, s.cnt.p, s.pstart.p);
    u64 total = scan_u32_u64(ctx, s.cnt.p, nf, s.offs.p);
    // a pull round reads every edge without atomics; measured on R-MAT it costs about
    // what pushing an eighth of the edges does
    if (form == WCC_AUTO && 8 * total >= (u64)ix.n) return wcc_pull_round(ctx, s, ix, nbr);
    fill_u32(ctx, s.counter.p, 1, 0u);
    if (total) {
        // 4 B neighbour id + 4 B label read + 4 B atomicMin per edge, frontier reads amortised
        DLG_LAUNCH(ctx, DLG_K_WCC_RELAX, 12.0 * total + 8.0 * nf, wcc_relax_k, grid_for(total, WR_TILE),
                   WR_T, 0, (const u32 *)s.flabel.p, nf, (const u32 *)s.pstart.p,
                   (const u64 *)s.offs.p, total, nbr, s.L.p, s.mark.p, round, s.nnode.p,
                   s.counter.p);
    }
    const u64 h = read_counter(ctx, s);
    if (h) {
        DLG_LAUNCH(ctx, DLG_K_WCC_RELAX, 12.0 * h, wcc_gather_k, sgrid(ctx, h), ctx->block_size, 0,
                   (const u32 *)s.nnode.p, h, (const u32 *)s.L.p, s.flabel.p);
    }
    s.fnode.swap(s.nnode);
    return h;
}

// One thread per join row of Δ ⋈ E (load-balanced like wcc_relax_k): row r
// of probe i gives node m = value of rows[r] at cc position nbr[r] and the
// candidate (m, label of Δ[i]); cc[nbr[r]] takes the lesser.  A value that is
// no key, or a cc tuple of another node, raises *bad.
__global__ __launch_bounds__(WR_T) void wcc_tuple_relax_k(const u64 *delta, u64 nd, const u32 *pstart,
                                                          const u64 *offs, u64 total, const u64 *rows,
                                                          const u32 *nbr, u64 ncc, u64 *cc, u32 *bad) {
    __shared__ u64 s_lo, s_hi;
    const u64 base = (u64)blockIdx.x * WR_TILE;
    if (threadIdx.x < WAVE) {   // the first wave finds the tile's probes
        const u64 last = (base + WR_TILE < total ? base + WR_TILE : total) - 1;
        const u64 lo = wave_upper_bound(offs, 0, nd, base) - 1;
        const u64 hi = wave_upper_bound(offs, lo, nd, last);
        if (threadIdx.x == 0) {
            s_lo = lo;
            s_hi = hi;
        }
    }
    __syncthreads();
    const u64 lo = s_lo, hi = s_hi;
#pragma unroll
    for (int r = 0; r < WR_I; r++) {
        const u64 o = base + (u64)r * WR_T + threadIdx.x;
        if (o < total) {
            const u64 i = upper_bound_u64(offs, lo, hi, o) - 1;
            const u64 row = (u64)pstart[i] + (o - offs[i]);
            const u32 g = nbr[row];
            const u64 t = tmake(tval(rows[row]), tval(delta[i]));
            if (g >= ncc) {
                *bad = 1u;
            } else {
                const u64 cur = cc[g];
                if (tkey(cur) != tkey(t)) *bad = 1u;
                else if (cur > t) atomicMin((unsigned long long *)&cc[g], (unsigned long long)t);
            }
        }
    }
}

u64 wcc_relax_tuples(dlg_ctx *ctx, const Index &ix, const u32 *nbr, const u64 *delta, u64 nd, u64 *cc, u64 ncc,
                     u64 *next) {
    if (nd == 0 || ncc == 0 || ix.n == 0) return 0;
    DBuf<u64> old(ctx, ncc);
    copy_u64(ctx, old.p, cc, ncc);
    JoinScratch js(ctx);
    const u64 total = join_count(ctx, ix, delta, nd, js);
    DBuf<u32> bad(ctx, 1);
    fill_u32(ctx, bad.p, 1, 0u);
    if (total)
        // 4 B group + 8 B row + 8 B cc read per join row (the atomic only when lower), Δ reads amortised
        DLG_LAUNCH(ctx, DLG_K_WCC_RELAX, 20.0 * total + 8.0 * nd, wcc_tuple_relax_k, grid_for(total, WR_TILE), WR_T,
                   0, delta, nd, (const u32 *)js.pstart.p, (const u64 *)js.offs.p, total, (const u64 *)ix.rows.p,
                   nbr, ncc, cc, bad.p);
    u32 hb = 0;
    ctx->read_words(bad.p, 1, &hb);
    if (hb) fail(DLG_INVALID_INPUT, "dlg_wcc_relax: a join row's node is not in cc (edges not symmetric, or cc "
                                    "not one tuple per key in key order)");
    // cc' keeps cc's node order, so both are sorted: Δ' = cc' minus cc
    return select(ctx, SEL_NOT_IN, cc, ncc, old.p, ncc, next);
}

void wcc_setup(dlg_ctx *ctx, WccState &s, u64 V) {
    s.V = V;
    s.L.ensure(V);
    s.mark.ensure(V);
    s.fnode.ensure(V);
    s.flabel.ensure(V);
    s.nnode.ensure(V);
    s.counter.ensure(4);
    if (V)
        DLG_LAUNCH(ctx, DLG_K_MISC, 16.0 * V, wcc_init_k, sgrid(ctx, V), ctx->block_size, 0, s.L.p, s.fnode.p,
                   s.flabel.p, s.mark.p, V);
}

// Frontier lists and marks, the labels left as they are.
static void wcc_lists(dlg_ctx *ctx, WccState &s, u64 V) {
    s.mark.ensure(V);
    s.fnode.ensure(V);
    s.flabel.ensure(V);
    s.nnode.ensure(V);
    fill_u32(ctx, s.mark.p, V, 0u);
}

// Components: returns #distinct labels, *largest, and the (label, 0) tuples in `out`.
u64 wcc_finalize(dlg_ctx *ctx, WccState &s, const Index &ix, DBuf<u64> &out, i64 *largest) {
    u64 V = s.V;
    *largest = -1;
    if (V == 0) return 0;
    DBuf<u32> ccount(ctx, V), flags(ctx, V);
    DBuf<u64> offs(ctx, V + 1);
    fill_u32(ctx, ccount.p, V, 0u);
    fill_u32(ctx, s.counter.p, 1, 0u);
    DLG_LAUNCH(ctx, DLG_K_WCC_FINAL, 12.0 * V, wcc_comp_count_k, grid_for(V, WA_TILE), WA_T, 0,
               (const u32 *)s.L.p, V, ccount.p);
    DLG_LAUNCH(ctx, DLG_K_WCC_FINAL, 8.0 * V, wcc_comp_flags_k, sgrid(ctx, V), ctx->block_size, 0,
               (const u32 *)ccount.p, V, flags.p, s.counter.p);
    u64 ncomp = scan_u32_u64(ctx, flags.p, V, offs.p);
    *largest = (i64)read_counter(ctx, s);
    out.ensure(ncomp ? ncomp : 1);
    DLG_LAUNCH(ctx, DLG_K_WCC_FINAL, 16.0 * V, wcc_emit_k, sgrid(ctx, V), ctx->block_size, 0,
               (const u32 *)flags.p, (const u64 *)offs.p, V, (const u64 *)ix.rows.p,
               (const u32 *)ix.gstart.p, out.p);
    return ncomp;
}

}  // namespace dlg

// =====================================================================
// Whole-graph rounds: for graphs of moderate size every round pulls every
// node from the labels of the round before (two label arrays in turn: exactly
// the Jacobi round) in ONE launch -- no frontier, no degree scan, no append,
// no label atomics.  Rounds are queued ahead of the host: kernel r publishes
// round r - 1's count, applies the stop rule to it and, when it fires, lets the
// kernels after it do nothing (round r itself writes the other array, so the
// labels of the last counted round stay in theirs).
// A thread takes a node of up to WD_THREAD edges, a wave one of up to WD_WAVE, a
// workgroup WD_SEG edges of a larger one (a hub's segments meet in an atomic
// minimum).
// Bound by the latency of start -> neighbour -> label (L2) for small graphs, by
// the label reads for large ones.
// Whole calls against the captured push rounds, which stay for `strategy` 2:
// 160,000 nodes, 355,000 edges, ~500 rounds 15.4 -> 2.0 ms (a round 4.6 us
// instead of 41); 12.4M nodes, 28.8M edges, 4,303 rounds 2,693 -> 344 ms;
// R-MAT 2^17 to 2^20 nodes 1.36 -> 0.82 and 4.3 -> 4.1 ms; a star of 200,000
// 1.0 -> 0.56 ms (1.1 with its hub in one workgroup).  Where they cost more than the captured
// rounds (many rounds of few nodes), those take over: see wcc_rounds_whole.
// Batches: 400 instances 2.8 -> 1.6 ms on the device.
namespace dlg {

constexpr int WD_T = 256, WD_SLOTS = 64, WD_SETS = 4, WD_LINE = 8;
constexpr u32 WD_THREAD = 16, WD_WAVE = 1024, WD_SEG = 8192;
constexpr int WD_DEPTH = 4;   // rounds queued ahead of the host
static_assert(WD_DEPTH + 2 <= dlg_ctx::MAPPED_SLOTS, "every queued round has a mapped slot of its own");

struct WdState {
    unsigned long long cnt[WD_SETS][WD_SLOTS][WD_LINE];   // lowered nodes, by round and slice
    u64 prev;    // |Δ| of the round before (wcc.cu:236-242)
    u32 done;    // the round that published the stop rule's firing, every instance's (0: not yet)
    u32 nmid, nhub;   // middle nodes, hub segments
};

// The batched form's instances (contiguous node ranges), each with its own
// stop rule: an instance's labels stay where its last round left them, in
// the array of that round's parity, and the end picks them from there.
struct WdInst {
    const u32 *of;       // each node's instance (null: one graph)
    u32 B;
    u32 *cnt;            // WD_SETS sets of B counts
    u32 *prev, *done, *iters;
};

// The nodes that a wave takes, and the segments (node, first edge) that a
// workgroup takes.
__global__ __launch_bounds__(WD_T) void wd_lists_k(const u32 *gstart, u64 V, u32 *mid, uint2 *hub, WdState *st) {
    const int lane = threadIdx.x & (WAVE - 1);
    const u64 stride = (u64)gridDim.x * WD_T, lim = (V + WAVE - 1) / WAVE * WAVE;   // whole waves iterate together
    for (u64 i = (u64)blockIdx.x * WD_T + threadIdx.x; i < lim; i += stride) {
        const u32 a = i < V ? gstart[i] : 0u, d = i < V ? gstart[i + 1] - a : 0u;
        const bool is_mid = d > WD_THREAD && d <= WD_WAVE;
        const u64 bm = __ballot(is_mid);
        u32 b = 0;
        if (lane == 0 && bm) b = atomicAdd(&st->nmid, (u32)__popcll(bm));
        b = (u32)__shfl((int)b, 0, WAVE);
        if (is_mid) mid[b + (u32)__popcll(bm & lanemask_lt())] = (u32)i;
        if (d > WD_WAVE) {
            u32 j = atomicAdd(&st->nhub, (d + WD_SEG - 1) / WD_SEG);
            for (u32 e = 0; e < d; e += WD_SEG) hub[j++] = make_uint2((u32)i, a + e);
        }
    }
}

// Identity labels in both arrays: a hub's segments lower a label of two rounds
// ago, which is never below the last one.
__global__ void wd_init_k(WdState *st, u32 *L, u32 *Ln, u64 V) {
    const u64 i0 = (u64)blockIdx.x * blockDim.x + threadIdx.x, stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = i0; i < V; i += stride) L[i] = Ln[i] = (u32)i;
    for (u64 i = i0; i < (u64)WD_SETS * WD_SLOTS * WD_LINE; i += stride) (&st->cnt[0][0][0])[i] = 0;
    if (i0 == 0) {
        st->prev = V;
        st->done = st->nmid = st->nhub = 0;
    }
}

__global__ void wd_sizes_k(const WdState *st, u64 *host, u64 seq) {
    if (threadIdx.x != 0) return;
    host[0] = st->nmid;
    host[1] = st->nhub;
    __threadfence_system();
    *(volatile u64 *)(host + dlg_ctx::MAPPED_SEQ) = seq;
    __threadfence_system();
}

__device__ __forceinline__ u32 wd_wave_min(u32 v) {
#pragma unroll
    for (int d = WAVE / 2; d > 0; d >>= 1) v = min(v, (u32)__shfl_xor((int)v, d, WAVE));
    return v;
}

// Nodes the threads lowered: into the round's count, by slice, or (instances)
// by the node's instance.
template <bool MULTI>
__device__ __forceinline__ void wd_count(WdState *st, const WdInst &in, u32 round, u32 wg, bool low, u32 inst, u32 *s_v) {
    const int lane = threadIdx.x & (WAVE - 1);
    if (MULTI) {
        wave_count_by_key(in.cnt + (u64)(round % WD_SETS) * in.B, inst, low);
        return;
    }
    const u32 c = (u32)__popcll(__ballot(low));
    if (lane == 0) s_v[threadIdx.x / WAVE] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        u32 t = 0;
        for (int w = 0; w < WD_T / WAVE; w++) t += s_v[w];
        if (t) atomicAdd(&st->cnt[round % WD_SETS][wg % WD_SLOTS][0], (unsigned long long)t);
    }
}

// Publishes round `round` - 1: the stop rule (wcc.cu:366-383) on its count, or
// on each instance's; host[0] = the nodes it lowered (of the instances left),
// host[1] = nothing is left to run.
template <bool MULTI>
__device__ __forceinline__ void wd_publish(WdState *st, const WdInst &in, u32 round, u64 *host, u64 seq) {
    __shared__ u32 s_live, s_low;
    if (MULTI) {
        if (threadIdx.x == 0) s_live = s_low = 0;
        __syncthreads();
        const u32 *cur = in.cnt + (u64)((round - 1) % WD_SETS) * in.B;
        u32 *next = in.cnt + (u64)((round + 1) % WD_SETS) * in.B;
        u32 live = 0, low = 0;
        for (u32 i = threadIdx.x; i < in.B; i += WD_T) {
            next[i] = 0;
            if (in.done[i]) continue;
            in.iters[i] = round - 1;
            if (cur[i] == in.prev[i]) {
                in.done[i] = 1;
            } else {
                live++;
                low += cur[i];
            }
            in.prev[i] = cur[i];
        }
        if (live) atomicAdd(&s_live, live);
        if (low) atomicAdd(&s_low, low);
        __syncthreads();
        if (threadIdx.x == 0) {
            if (s_live == 0 && !st->done) st->done = round;
            host[0] = s_low;
            host[1] = st->done != 0;
        }
    } else if (threadIdx.x < WAVE) {   // WD_SLOTS == WAVE: a slice per lane
        u64 c = st->cnt[(round - 1) % WD_SETS][threadIdx.x][0];
        st->cnt[(round + 1) % WD_SETS][threadIdx.x][0] = 0;
#pragma unroll
        for (int d = WAVE / 2; d > 0; d >>= 1) c += __shfl_xor(c, d, WAVE);
        if (threadIdx.x == 0) {
            if (c == st->prev && !st->done) st->done = round;
            host[0] = c;
            host[1] = st->done != 0;
            st->prev = c;
        }
    }
    if (threadIdx.x == 0) {
        __threadfence_system();
        *(volatile u64 *)(host + dlg_ctx::MAPPED_SEQ) = seq;
        __threadfence_system();
    }
}

// Round `round` from L into Ln, the round before published first (or only
// the publication).  Workgroups: the publisher, the nodes by thread, the
// middle nodes by wave, the hubs' segments by workgroup.
template <bool MULTI>
__global__ __launch_bounds__(WD_T) void wd_round_k(const u32 *gstart, const u32 *nbr, u64 V, const u32 *L, u32 *Ln,
                                                   const u32 *mid, u32 nmid, const uint2 *hub, WdState *st, WdInst in,
                                                   u32 round, int publish_only, u64 *host, u64 seq) {
    __shared__ u32 s_v[WD_T / WAVE];
    const int lane = threadIdx.x & (WAVE - 1), wv = threadIdx.x / WAVE;
    if (blockIdx.x == 0) {
        if (round > 1) wd_publish<MULTI>(st, in, round, host, seq);
        return;
    }
    // its own publisher may set `done` meanwhile, which must not part a workgroup's waves: earlier rounds' only
    const u32 stop = *(volatile const u32 *)&st->done;
    if (publish_only || (stop && stop < round)) return;
    const u32 wg = blockIdx.x - 1, nthr = (u32)((V + WD_T - 1) / WD_T), nwav = (nmid + WD_T / WAVE - 1) / (WD_T / WAVE);
    bool low = false;   // this thread lowered a node, of instance `inst`
    u32 inst = 0;
    if (wg < nthr) {
        const u64 i = (u64)wg * WD_T + threadIdx.x;
        if (i < V) {
            const u32 a = gstart[i], d = gstart[i + 1] - a;
            if (MULTI) inst = in.of[i];
            if (d <= WD_THREAD && !(MULTI && in.done[inst])) {
                const u32 old = L[i];
                u32 m = old;
                for (u32 e = 0; e < d; e += 4) {   // four neighbours in flight (a lane past the end reads the last again)
                    u32 v[4];
#pragma unroll
                    for (u32 k = 0; k < 4; k++) v[k] = nbr[a + min(e + k, d - 1)];
#pragma unroll
                    for (u32 k = 0; k < 4; k++) m = min(m, L[v[k]]);
                }
                Ln[i] = m;
                low = m < old;
            }
        }
    } else if (wg < nthr + nwav) {
        const u32 j = (wg - nthr) * (WD_T / WAVE) + (u32)wv;
        if (j < nmid) {
            const u32 i = mid[j], a = gstart[i], d = gstart[i + 1] - a;
            if (MULTI) inst = in.of[i];
            if (!(MULTI && in.done[inst])) {   // wave-uniform
                u32 m = 0xffffffffu;
                for (u32 e = (u32)lane; e < d; e += WAVE) m = min(m, L[nbr[a + e]]);
                m = wd_wave_min(m);
                if (lane == 0) {
                    const u32 old = L[i];
                    m = min(m, old);
                    Ln[i] = m;
                    low = m < old;
                }
            }
        }
    } else {
        const uint2 h = hub[wg - nthr - nwav];
        const u32 i = h.x, end = min(h.y + WD_SEG, gstart[i + 1]);
        if (MULTI) {   // one reading for the workgroup: the flag may be set while it runs
            inst = in.of[i];
            if (threadIdx.x == 0) s_v[0] = in.done[inst];
            __syncthreads();
            const bool fin = s_v[0] != 0;
            __syncthreads();
            if (fin) return;
        }
        u32 m = 0xffffffffu;
        for (u32 e = h.y + threadIdx.x; e < end; e += 4 * WD_T) {
            u32 v[4];
#pragma unroll
            for (u32 k = 0; k < 4; k++) v[k] = nbr[min(e + k * WD_T, end - 1)];
#pragma unroll
            for (u32 k = 0; k < 4; k++) m = min(m, L[v[k]]);
        }
        m = wd_wave_min(m);
        if (lane == 0) s_v[wv] = m;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int w = 1; w < WD_T / WAVE; w++) m = min(m, s_v[w]);
            const u32 old = L[i];
            // the node's first segment to go below its last label counts it
            low = atomicMin(&Ln[i], min(m, old)) >= old && m < old;
        }
        __syncthreads();   // s_v is rewritten below
    }
    wd_count<MULTI>(st, in, round, wg, low, inst, s_v);
}

// Each node's instance (vstart[i] <= v < vstart[i + 1]); the instances' state.
__global__ void wd_inst_k(const u32 *vstart, WdInst in, u64 V, u32 *of) {
    const u64 i0 = (u64)blockIdx.x * blockDim.x + threadIdx.x, stride = (u64)gridDim.x * blockDim.x;
    for (u64 v = i0; v < V; v += stride) {
        u32 a = 0, b = in.B;
        while (b - a > 1) {
            const u32 m = (a + b) >> 1;
            if (vstart[m] <= (u32)v) a = m; else b = m;
        }
        of[v] = a;
    }
    for (u64 i = i0; i < (u64)WD_SETS * in.B; i += stride) in.cnt[i] = 0;
    for (u64 i = i0; i < in.B; i += stride) {
        in.prev[i] = vstart[i + 1] - vstart[i];
        in.done[i] = in.iters[i] = 0;
    }
}
// Rounds from labels L whose last round lowered `prev` nodes: both arrays hold them.
__global__ void wd_again_k(WdState *st, const u32 *L, u32 *Ln, u64 V, u64 prev) {
    const u64 i0 = (u64)blockIdx.x * blockDim.x + threadIdx.x, stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = i0; i < V; i += stride) Ln[i] = L[i];
    for (u64 i = i0; i < (u64)WD_SETS * WD_SLOTS * WD_LINE; i += stride) (&st->cnt[0][0][0])[i] = 0;
    if (i0 == 0) {
        st->prev = prev;
        st->done = 0;
    }
}
// The instances' labels after `rounds` rounds to L (those of its last round where the rule has fired),
// and the nodes that the last round lowered in the others.
__global__ __launch_bounds__(WA_T) void wd_export_k(u32 *L, const u32 *Ln, u64 V, WdInst in, u32 rounds, u32 *node, u32 *label,
                                                    u32 *count) {
    __shared__ u32 s_cnt[WA_I * WA_T / WAVE + 1];
    const u64 base = (u64)blockIdx.x * WA_TILE;
    bool app[WA_I];
    u32 l[WA_I], slot[WA_I];
#pragma unroll
    for (int r = 0; r < WA_I; r++) {
        const u64 i = base + (u64)r * WA_T + threadIdx.x;
        app[r] = false;
        l[r] = 0;
        if (i < V) {
            const u32 inst = in.of[i], a = L[i], b = Ln[i];
            const bool fin = in.done[inst] != 0, odd = ((fin ? in.iters[inst] : rounds) & 1u) != 0;
            l[r] = odd ? b : a;
            app[r] = !fin && l[r] < (odd ? a : b);
            L[i] = l[r];
        }
    }
    block_append<WA_T, WA_I>(app, count, s_cnt, slot);
#pragma unroll
    for (int r = 0; r < WA_I; r++)
        if (app[r]) {
            node[slot[r]] = (u32)(base + (u64)r * WA_T + threadIdx.x);
            label[slot[r]] = l[r];
        }
}
// The labels of each node's instance's last round.
__global__ void wd_pick_k(u32 *L, const u32 *Ln, u64 V, WdInst in) {
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 v = (u64)blockIdx.x * blockDim.x + threadIdx.x; v < V; v += stride)
        if (in.iters[in.of[v]] & 1u) L[v] = Ln[v];
}

// ---------------------------------------------------------- one workgroup's rounds
// The whole run of a small graph by one workgroup, a round two barriers instead of a
// launch: the labels in LDS twice, a thread's consecutive edges (their other ends, and a bit
// for each that begins a node) and its nodes' labels in registers.  A round reads the label of
// every edge's end, all of a thread's in flight, and gives each node's least to the new labels.
// Bound by one CU's LDS: whole calls against launched rounds, a 40 x 40 grid (1,522 nodes, 76
// rounds) 511 -> 375 us, 60 x 60 679 -> 532, 100 random nodes 246 -> 212; from 16,000 edges
// on as fast (a path of 8,000, 8,002 rounds, 33.0 and 32.9 ms).
constexpr int WO_T = 1024, WO_E = 16, WO_N = 16;   // threads; edges and nodes a thread at most
constexpr u64 WO_MAX = (u64)WO_T * WO_E;
static bool wo_takes(u64 V, u64 ne) { return ne <= WO_MAX && V <= (u64)WO_T * WO_N; }

__global__ __launch_bounds__(WO_T) void wo_rounds_k(const u32 *gstart, const u32 *nbr, u32 V, u32 ne, int max_it, u32 *L,
                                                    u64 *host, u64 seq) {
    __shared__ u32 A[WO_T * WO_N], B[WO_T * WO_N], s_cnt[2];
    u32 lab[WO_N];   // of nodes j * WO_T + threadIdx.x
#pragma unroll
    for (int j = 0; j < WO_N; j++) {
        const u32 i = (u32)j * WO_T + threadIdx.x;
        lab[j] = i;
        if (i < V) A[i] = B[i] = i;
    }
    if (threadIdx.x < 2) s_cnt[threadIdx.x] = 0;
    const u32 per = (ne + WO_T - 1) / WO_T, e0 = min(threadIdx.x * per, ne), n = min(per, ne - e0);
    u32 own = 0;   // the node of edge e0
    for (u32 hi = V; hi - own > 1;) {
        const u32 m = (own + hi) >> 1;
        if (gstart[m] <= e0) own = m; else hi = m;
    }
    u32 nb[WO_E], first = 0;
    {
        u32 m = own;
#pragma unroll
        for (int k = 0; k < WO_E; k++) {
            nb[k] = (u32)k < n ? nbr[e0 + (u32)k] : 0u;
            if (k && (u32)k < n && gstart[m + 1] == e0 + (u32)k) {   // every node has an edge
                first |= 1u << k;
                m++;
            }
        }
    }
    __syncthreads();
    u32 prev = V;   // wcc.cu:236-242
    int it = 0;
    while (true) {
        if (n) {
            u32 v[WO_E];
#pragma unroll
            for (int k = 0; k < WO_E; k++)
                if ((u32)k < per) v[k] = A[nb[k]];   // block-uniform; past the end: node 0's, not used
            u32 m = own, cur = 0xffffffffu;
#pragma unroll
            for (int k = 0; k < WO_E; k++) {
                if ((u32)k >= n) continue;
                if ((first >> k) & 1u) {
                    atomicMin(&B[m++], cur);
                    cur = v[k];
                } else {
                    cur = min(cur, v[k]);
                }
            }
            atomicMin(&B[m], cur);
        }
        __syncthreads();
        if (threadIdx.x == 0) s_cnt[(it + 1) & 1] = 0;   // read by all before the barrier above
        u32 c = 0;
#pragma unroll
        for (int j = 0; j < WO_N; j++) {
            const u32 i = (u32)j * WO_T + threadIdx.x;
            if (i >= V) continue;
            const u32 b = B[i];
            if (b < lab[j]) {
                lab[j] = b;
                A[i] = b;
                c++;
            }
        }
#pragma unroll
        for (int d = WAVE / 2; d > 0; d >>= 1) c += (u32)__shfl_xor((int)c, d, WAVE);
        if (threadIdx.x % WAVE == 0 && c) atomicAdd(&s_cnt[it & 1], c);
        __syncthreads();
        c = s_cnt[it & 1];
        it++;
        if (c == prev || (max_it > 0 && it >= max_it)) break;   // block-uniform; wcc.cu:366-383
        prev = c;
    }
    for (u32 i = threadIdx.x; i < V; i += WO_T) L[i] = A[i];
    if (threadIdx.x == 0) {
        host[0] = (u64)it;
        __threadfence_system();
        *(volatile u64 *)(host + dlg_ctx::MAPPED_SEQ) = seq;
        __threadfence_system();
    }
}

}  // namespace dlg

// =====================================================================
// Graph-captured rounds.  For long runs with small frontiers the eager
// round costs more in launches and host synchronisation than in work.
// Here every size lives in device memory (WccDev), every kernel has a
// fixed grid sized for the whole graph and exits early past the live size,
// the stop rule runs on the device, and KR rounds (frontier buffers in
// ping-pong) are captured once into a hipGraph that the host replays,
// reading back one flag per replay.  No memset nodes: counters are cleared
// by kernels.  Four kernels a round: the frontier's degrees and label
// snapshot, their scan, the relax, the stop rule.
namespace dlg {

struct WccDev {
    u64 nf;      // live frontier size
    u64 total;   // edges leaving the frontier
    u32 count;   // next frontier size (append counter)
    u32 done;    // the stop rule fired
    u32 it;      // rounds run
    u32 max_it;  // 0 = none
    u64 prev;    // |Δ| of the previous round (wcc.cu:236-242, 366-383)
};

constexpr int GW_T = 256, GW_I = 8, GW_TILE = GW_T * GW_I;

// Degrees of the frontier's nodes and their block sums; each node's label is
// read here too, after the previous round's relax: the snapshot its edges
// carry this round (Jacobi).
__global__ __launch_bounds__(GW_T) void gw_degree_scan_k(const u32 *fnode, const u32 *gstart, const u32 *L,
                                                         u32 *flabel, u32 *cnt, u32 *pstart, u64 *bsum,
                                                         const WccDev *st) {
    __shared__ u64 sc[GW_T / WAVE + 1];
    const u64 nf = st->done ? 0 : st->nf;
    const u64 base = (u64)blockIdx.x * GW_TILE + (u64)threadIdx.x * GW_I;
    u64 s = 0;
#pragma unroll
    for (int i = 0; i < GW_I; i++) {
        u64 j = base + i;
        if (j < nf) {
            u32 v = fnode[j];
            u32 a = gstart[v];
            u32 c = gstart[v + 1] - a;
            cnt[j] = c;
            pstart[j] = a;
            flabel[j] = L[v];
            s += c;
        }
    }
    u64 tot;
    block_exclusive_scan<u64>(s, sc, &tot);
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// Offsets of the frontier's edges: each workgroup adds the block sums before
// its own (read and summed by the whole workgroup) to a scan of its degrees;
// the last workgroup also writes the round's edge total.
__global__ __launch_bounds__(GW_T) void gw_scan_apply_k(const u32 *cnt, const u64 *bsum, u64 *offs, WccDev *st) {
    __shared__ u64 sc[GW_T / WAVE + 1];
    const u64 nf = st->done ? 0 : st->nf;
    const bool last = blockIdx.x == gridDim.x - 1;
    const u64 base = (u64)blockIdx.x * GW_TILE + (u64)threadIdx.x * GW_I;
    if ((u64)blockIdx.x * GW_TILE >= nf && !last) return;   // block-uniform: no frontier nodes here
    u64 p = 0;
    for (u64 i = threadIdx.x; i < blockIdx.x; i += GW_T) p += bsum[i];
    u64 pre;
    block_exclusive_scan<u64>(p, sc, &pre);
    __syncthreads();   // sc is reused
    if (last && threadIdx.x == 0) st->total = pre + bsum[blockIdx.x];   // 0 when the rule has fired
    u32 v[GW_I];
    u64 s = 0;
#pragma unroll
    for (int i = 0; i < GW_I; i++) {
        v[i] = base + i < nf ? cnt[base + i] : 0;
        s += v[i];
    }
    u64 ex = block_exclusive_scan<u64>(s, sc, nullptr) + pre;
#pragma unroll
    for (int i = 0; i < GW_I; i++) {
        if (base + i < nf) offs[base + i] = ex;
        ex += v[i];
    }
}

__global__ __launch_bounds__(WR_T) void gw_relax_k(const u32 *flabel, const u32 *pstart, const u64 *offs,
                                                   const u32 *nbr, u32 *L, u32 *mark, u32 *next_node,
                                                   WccDev *st) {
    __shared__ u64 s_lo, s_hi;
    __shared__ u32 s_cnt[WR_I * WR_T / WAVE + 1];
    __shared__ TileStarts ts;
    const u64 total = st->total, nf = st->nf;
    const u64 base = (u64)blockIdx.x * WR_TILE;
    if (st->done || base >= total) return;   // block-uniform
    const u32 round = st->it + 1;
    tile_starts_clear(ts);
    if (threadIdx.x < WAVE) {   // the first wave finds the tile's frontier nodes
        const u64 last = (base + WR_TILE < total ? base + WR_TILE : total) - 1;
        const u64 lo = wave_upper_bound(offs, 0, nf, base) - 1;
        const u64 hi = wave_upper_bound(offs, lo, nf, last);
        if (threadIdx.x == 0) {
            s_lo = lo;
            s_hi = hi;
        }
    }
    __syncthreads();
    const u64 lo = s_lo, hi = s_hi;
    tile_starts_set<WR_T>(ts, offs, lo, hi, base);   // frontier nodes have edges: offsets rise strictly
    bool app[WR_I];
    u32 m[WR_I], slot[WR_I];
#pragma unroll
    for (int r = 0; r < WR_I; r++) {
        u64 o = base + (u64)r * WR_T + threadIdx.x;
        app[r] = false;
        m[r] = 0;
        if (o < total) {
            const u64 i = lo + tile_owner(ts, (u32)(r * WR_T) + threadIdx.x);
            m[r] = nbr[(u64)pstart[i] + (o - offs[i])];
            u32 l = flabel[i];
            if (L[m[r]] > l) {
                u32 old = atomicMin(&L[m[r]], l);
                if (old > l) app[r] = atomicExch(&mark[m[r]], round) != round;
            }
        }
    }
    block_append<WR_T, WR_I>(app, &st->count, s_cnt, slot);
#pragma unroll
    for (int r = 0; r < WR_I; r++)
        if (app[r]) next_node[slot[r]] = m[r];
}

// The reference's stop rule, on the device: count the round, stop when two
// consecutive delta sizes are equal.  The append counter is cleared for the
// next round.
__global__ void gw_end_k(WccDev *st) {
    if (threadIdx.x != 0 || blockIdx.x != 0 || st->done) return;
    u64 cur = st->count;
    st->count = 0;
    st->it += 1;
    st->nf = cur;
    if (cur == st->prev || (st->max_it && st->it >= st->max_it)) st->done = 1;
    else st->prev = cur;
}

static void gw_capture_round(dlg_ctx *ctx, WccState &s, const Index &ix, const u32 *nbr, u64 V, u64 E,
                             WccDev *st, u32 *fnode, u32 *flabel, u32 *nnode, u64 *bsum) {
    const unsigned gb = grid_for(V, GW_TILE);   // bsum holds gb block sums
    hipLaunchKernelGGL(gw_degree_scan_k, dim3(gb), dim3(GW_T), 0, ctx->stream, (const u32 *)fnode,
                       (const u32 *)ix.gstart.p, (const u32 *)s.L.p, flabel, s.cnt.p, s.pstart.p, bsum,
                       (const WccDev *)st);
    hipLaunchKernelGGL(gw_scan_apply_k, dim3(gb), dim3(GW_T), 0, ctx->stream, (const u32 *)s.cnt.p,
                       (const u64 *)bsum, s.offs.p, st);
    hipLaunchKernelGGL(gw_relax_k, dim3(grid_for(E, WR_TILE)), dim3(WR_T), 0, ctx->stream,
                       (const u32 *)flabel, (const u32 *)s.pstart.p, (const u64 *)s.offs.p, nbr, s.L.p,
                       s.mark.p, nnode, st);
    hipLaunchKernelGGL(gw_end_k, dim3(1), dim3(64), 0, ctx->stream, st);
}

__global__ void gw_start_k(WccDev *st, WccDev h) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *st = h;
}

typedef std::chrono::steady_clock WallClock;
static double wall_us(WallClock::time_point t0) { return std::chrono::duration<double, std::micro>(WallClock::now() - t0).count(); }

// A captured graph of `kr` rounds (even) on the labels in L, replayed until `go` says no.
struct GwRounds {
    dlg_ctx *ctx;
    u32 *L;
    DBuf<u32> nlabel;
    DBuf<u64> bsum, stbuf;
    WccDev *st;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;

    // s: fnode, flabel, nnode and mark are there (wcc_setup, wcc_lists)
    GwRounds(dlg_ctx *c, WccState &s, const Index &ix, const u32 *nbr, u64 ne, int kr)
        : ctx(c), L(s.L.p), nlabel(c, s.V), bsum(c, (s.V + GW_TILE - 1) / GW_TILE + 1), stbuf(c, (sizeof(WccDev) + 7) / 8) {
        const u64 V = s.V;
        s.cnt.ensure(V);
        s.pstart.ensure(V);
        s.offs.ensure(V + 1);
        st = (WccDev *)stbuf.p;
        if (kr < 2) kr = 2;
        kr &= ~1;
        const bool prof = ctx->prof;
        ctx->prof = false;
        HIPCHK(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
        for (int r = 0; r < kr; r++) {
            if (r % 2 == 0)
                gw_capture_round(ctx, s, ix, nbr, V, ne, st, s.fnode.p, s.flabel.p, s.nnode.p, bsum.p);
            else
                gw_capture_round(ctx, s, ix, nbr, V, ne, st, s.nnode.p, nlabel.p, s.fnode.p, bsum.p);
        }
        const hipError_t ce = hipStreamEndCapture(ctx->stream, &graph);
        ctx->prof = prof;
        HIPCHK(ce);
        const hipError_t ie = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        if (ie != hipSuccess) {
            (void)hipGraphDestroy(graph);
            HIPCHK(ie);
        }
    }
    GwRounds(const GwRounds &) = delete;
    ~GwRounds() {
        (void)hipGraphExecDestroy(exec);
        (void)hipGraphDestroy(graph);
    }
    // From the nf nodes in fnode, lowered by round `it`, which follow a round that lowered `prev`.
    // go: whether to replay again, given what a round of the last replay took (us).
    template <typename F>
    WccDev run(u64 nf, u64 prev, int it, int max_it, F go) {
        WccDev h;
        std::memset(&h, 0, sizeof(h));
        h.nf = nf;
        h.prev = prev;
        h.it = (u32)it;
        h.max_it = (u32)(max_it > 0 ? max_it : 0);
        DLG_LAUNCH(ctx, DLG_K_MISC, 0.0, gw_start_k, 1, 64, 0, st, h);
        while (true) {
            const auto t0 = WallClock::now();
            const u32 before = h.it;
            if (ctx->prof) ctx->prof_begin();
            HIPCHK(hipGraphLaunch(exec, ctx->stream));
            if (ctx->prof) ctx->prof_end(DLG_K_WCC_RELAX, 0.0);
            static_assert(sizeof(WccDev) <= 8 * dlg_ctx::MAPPED_SEQ, "the state fits a mapped slot");
            ctx->read_words((const u32 *)st, (int)(sizeof(WccDev) / 4), &h);
            if (h.done || !go(wall_us(t0) / (double)(h.it - before))) return h;
        }
    }
};

// Runs the rounds of wcc_solve with captured graphs of `kr` rounds (even).
// Returns the iteration count; the labels are left in s.L.
int wcc_rounds_graph(dlg_ctx *ctx, WccState &s, const Index &ix, const u32 *nbr, u64 ne, int max_it,
                     int kr) {
    const u64 V = s.V;
    if (V == 0) return 1;   // empty graph: the first round already sees 0 == 0
    GwRounds g(ctx, s, ix, nbr, ne, kr);
    return (int)g.run(V, V, 0, max_it, [](double) { return true; }).it;
}

// ------------------------------------------------------ whole-graph rounds, run
// A pull of the whole graph costs what the graph costs, however few nodes a round lowers:
// a core with a long tail (R-MAT of 2^20 nodes and a path of 3,000 behind it) took 146, 292
// and 448 ms with 8, 17 and 31 million edges, by captured push rounds 82, 85 and 85.  So the
// pulls are left for those once they have cost WD_LEAVE_US more than those would have (81, 80
// and 83 ms), and taken up again where the pushes turn out to take longer.
// A pull's time is taken from the rounds themselves, and from the edges where they say more
// (something else may hold them up): at random 18, 46, 97 and 149 us at 2.1, 6.3, 16.8 and 31
// million, in grids half of that.  A push round's comes from the nodes lowered: 15 us up to a hundred,
// 27 at 1,500, 36 at 13,000, 40 at 130,000, 95 at 1,000,000 of one edge on and one back.
constexpr double WD_LEAVE_US = 250.0;   // a few pulls; the switch and the pulls queued cost as much again
static double wd_pull_us(u64 ne) { return 5.0 + (double)ne / 190e3; }
static double gw_push_us(u64 nodes) { return 15.0 + std::min((double)nodes / 256.0, 25.0) + (double)nodes / 16384.0; }
// A round that wcc_batch_rounds launches by itself: 77 us at least.
static double wd_batch_push_us(u64 nodes, u32 B) { return 80.0 + 0.003 * (double)B + (double)nodes / 8192.0; }

int wcc_rounds_whole(dlg_ctx *ctx, WccState &s, u64 V, const Index &ix, const u32 *nbr, int max_it, const u32 *vstart,
                     u32 B, std::vector<u32> *iters, WccRest *rest) {
    s.V = V;
    if (iters) iters->assign(B, 1);
    if (V == 0) return 1;   // empty graph: the first round already sees 0 == 0
    s.L.ensure(V);
    s.counter.ensure(4);
    if (!vstart && wo_takes(V, ix.n)) {
        const u64 seq = ++ctx->mapped_seq;
        DLG_LAUNCH(ctx, DLG_K_WCC_RELAX, 8.0 * ix.n + 16.0 * V, wo_rounds_k, 1, WO_T, 0, (const u32 *)ix.gstart.p, nbr, (u32)V,
                   (u32)ix.n, max_it, s.L.p, ctx->mapped_dev(seq), seq);
        ctx->wait_mapped(seq);
        return (int)ctx->mapped_host(seq)[0];
    }
    static_assert(WD_SLOTS == WAVE, "the publisher's wave sums a slice per lane");
    DBuf<u64> stbuf(ctx, (sizeof(WdState) + 7) / 8);
    WdState *st = (WdState *)stbuf.p;
    s.Ln.ensure(V);
    DLG_LAUNCH(ctx, DLG_K_MISC, 8.0 * V, wd_init_k, sgrid(ctx, V), ctx->block_size, 0, st, s.L.p, s.Ln.p, V);
    DBuf<u32> mid(ctx, ix.n / WD_THREAD + 1);
    DBuf<uint2> hub(ctx, ix.n / WD_WAVE + ix.n / WD_SEG + 1);
    DLG_LAUNCH(ctx, DLG_K_MISC, 4.0 * V, wd_lists_k, (unsigned)std::min<u64>((V + WD_T - 1) / WD_T, (u64)ctx->num_cus * 8),
               WD_T, 0, (const u32 *)ix.gstart.p, V, mid.p, hub.p, st);
    WdInst in{nullptr, B, nullptr, nullptr, nullptr, nullptr};
    DBuf<u32> of(ctx), ist(ctx);
    if (vstart) {
        of.ensure(V);
        ist.ensure((u64)(WD_SETS + 3) * B);
        in.of = of.p;
        in.cnt = ist.p;
        in.prev = ist.p + (u64)WD_SETS * B;
        in.done = in.prev + B;
        in.iters = in.done + B;
        DLG_LAUNCH(ctx, DLG_K_MISC, 4.0 * V, wd_inst_k, sgrid(ctx, V), ctx->block_size, 0, vstart, in, V, of.p);
    }
    u64 seq = ++ctx->mapped_seq;
    DLG_LAUNCH(ctx, DLG_K_MISC, 0.0, wd_sizes_k, 1, 64, 0, (const WdState *)st, ctx->mapped_dev(seq), seq);
    ctx->wait_mapped(seq);
    const u32 nmid = (u32)ctx->mapped_host(seq)[0], nhub = (u32)ctx->mapped_host(seq)[1];
    const unsigned g = 1u + (unsigned)((V + WD_T - 1) / WD_T) + (nmid + WD_T / WAVE - 1) / (WD_T / WAVE) + nhub;
    std::deque<u64> q;   // sequence numbers of the rounds not read yet
    u32 *buf[2];         // a stretch's round r leaves its labels in buf[r & 1]
    int launched = 0;    // rounds of the stretch
    auto launch = [&](bool publish_only) {
        const u32 r = (u32)launched + 1;
        seq = r > 1 ? ++ctx->mapped_seq : 0;   // round 1 has no round before it
        auto go = [&](auto kern) {
            // 4 B neighbour + 4 B label per edge; a start and two labels per node
            DLG_LAUNCH(ctx, DLG_K_WCC_RELAX, publish_only ? 0.0 : 8.0 * ix.n + 16.0 * V, kern, publish_only ? 1u : g, WD_T,
                       0, (const u32 *)ix.gstart.p, nbr, V, (const u32 *)buf[(r - 1) & 1], buf[r & 1],
                       (const u32 *)mid.p, nmid, (const uint2 *)hub.p, st, in, r, publish_only ? 1 : 0,
                       ctx->mapped_dev(seq), seq);
        };
        if (vstart) go(wd_round_k<true>);
        else go(wd_round_k<false>);
        if (r > 1) q.push_back(seq);
        if (!publish_only) launched++;
    };
    const double pull_most = 1.5 * wd_pull_us(ix.n);
    double pull_us = pull_most, leave_us = WD_LEAVE_US;
    bool may_leave = !vstart || rest;
    std::unique_ptr<GwRounds> push;
    auto end_push = [&]() {   // as much memory for what follows as without it
        push.reset();
        for (DBuf<u32> *b : {&s.mark, &s.fnode, &s.flabel, &s.nnode, &s.cnt, &s.pstart}) b->release();
        s.offs.release();
    };
    int it = 0;   // rounds before the stretch
    while (true) {
        buf[0] = s.L.p;
        buf[1] = s.Ln.p;
        launched = 0;
        int seen = 0;
        u64 low = 0;
        double lost = 0.0;
        bool fin = false, closing = false;
        auto t0 = WallClock::now();   // of the last round seen
        while (true) {
            while (!closing && launched < seen + 1 + WD_DEPTH && (max_it <= 0 || it + launched < max_it)) launch(false);
            if (q.empty()) launch(true);   // nothing behind the last round publishes it
            ctx->wait_mapped(q.front());
            const volatile u64 *m = ctx->mapped_host(q.front());
            low = m[0];
            fin = m[1] != 0;
            q.pop_front();
            seen++;
            fin = fin || (max_it > 0 && it + seen >= max_it);
            if (fin || (closing && seen == launched)) break;
            if (seen > 1) pull_us = 0.75 * pull_us + 0.25 * std::min(wall_us(t0), pull_most);   // the rounds are queued: one's time
            t0 = WallClock::now();
            lost = std::max(0.0, lost + pull_us - (vstart ? wd_batch_push_us(low, B) : gw_push_us(low)));
            closing = closing || (may_leave && lost >= leave_us);
        }
        it += seen;
        if (vstart) {
            if (fin) {
                DLG_LAUNCH(ctx, DLG_K_MISC, 12.0 * V, wd_pick_k, sgrid(ctx, V), ctx->block_size, 0, s.L.p, (const u32 *)s.Ln.p,
                           V, in);
            } else {
                wcc_lists(ctx, s, V);
                fill_u32(ctx, s.counter.p, 1, 0u);
                DLG_LAUNCH(ctx, DLG_K_MISC, 16.0 * V, wd_export_k, grid_for(V, WA_TILE), WA_T, 0, s.L.p, (const u32 *)s.Ln.p, V,
                           in, (u32)it, s.fnode.p, s.flabel.p, s.counter.p);
                rest->left = true;
                rest->nf = low;
                rest->prev.resize(B);
                rest->done.resize(B);
                HIPCHK(hipMemcpyAsync(rest->prev.data(), in.prev, 4 * (size_t)B, hipMemcpyDeviceToHost, ctx->stream));
                HIPCHK(hipMemcpyAsync(rest->done.data(), in.done, 4 * (size_t)B, hipMemcpyDeviceToHost, ctx->stream));
                s.Ln.release();   // read by what is queued; the pool is the stream's own
            }
            HIPCHK(hipMemcpyAsync(iters->data(), in.iters, 4 * (size_t)B, hipMemcpyDeviceToHost, ctx->stream));
            ctx->sync();
            return it;
        }
        if (seen & 1) s.L.swap(s.Ln);   // the last round's labels in L, the one before's in Ln
        if (fin) break;
        if (!push) {
            try {
                wcc_lists(ctx, s, V);
                push.reset(new GwRounds(ctx, s, ix, nbr, ix.n, 16));
            } catch (const Error &e) {   // pulls need less
                if (e.status != DLG_OUT_OF_MEMORY) throw;
                may_leave = false;
                end_push();
            }
        }
        if (push) {
            fill_u32(ctx, s.counter.p, 1, 0u);
            DLG_LAUNCH(ctx, DLG_K_MISC, 16.0 * V, wcc_changed_k, grid_for(V, WA_TILE), WA_T, 0, s.Ln.p, (const u32 *)s.L.p, V,
                       s.fnode.p, s.flabel.p, s.counter.p);   // both arrays hold the last labels now
            int replays = 0;
            const WccDev h = push->run(low, low, it, max_it, [&](double us) { return replays++ == 0 || us <= pull_us; });   // the first one sets up
            it = (int)h.it;
            if (s.L.p != push->L) s.L.swap(s.Ln);
            if (h.done) break;
            low = h.prev;
            leave_us *= 8.0;   // rounds that grew again: the next time costs as much
        }
        DLG_LAUNCH(ctx, DLG_K_MISC, 8.0 * V, wd_again_k, sgrid(ctx, V), ctx->block_size, 0, st, (const u32 *)s.L.p, s.Ln.p, V, low);
    }
    if (push) end_push();
    return it;
}

}  // namespace dlg
