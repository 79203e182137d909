// k_tcdense.hip -- TC rounds as row ORs over maps of moderate width.
//
// With the full relation F as a row-major map (row = a path's end z, column
// = its source x: tuple order), and the round's new tuples as a second map D
// of the same shape, a TC round (tc.cu:140-314)
//     N = { (w, x) : (z, x) in D, (z, w) in E } \ F ;  F = F u N ;  D = N
// is, for every row w,
//     N row w = (OR of D row z over the predecessors z of w) & ~(F row w):
// whole words are combined instead of single join rows, nothing is expanded,
// hashed or appended, and the row's owner is the only writer of F row w and
// N row w, so there are no atomics on the maps.  F lies in tuple order and is
// read out as it lies.
//
// A task is one row's chunk of 64 words (2,048 sources) and takes 16 lanes (a
// uint4 each: 256 contiguous bytes per predecessor).  D has a flag per task:
// a task reads only its predecessors' flagged chunks, four in flight, and
// leaves its own flag, so rounds with few new tuples read little more than
// the flags.  Rows with more than TD_LONG predecessors (hubs) are taken by a
// whole workgroup per chunk instead.
//
// The cost of a round is bounded by (edges + 3 rows) * row bytes whatever the
// tuples: small enough for maps up to TD_MAX_W ids wide, whose three maps
// (100 MB) stay in the last-level cache; a wider map's rounds touch too few
// of a row's words at a time, and the row kernel of k_tcrows.hip takes them.
// Bound by the latency of dependent reads (list, flag, row) at small sizes
// and by the cache's bandwidth at large ones.
// Measured against the row kernel with its compaction and index build (whole
// call): 437 ids, 700 edges 1.13 -> 0.31 ms (a round 4.7 us; it was 14; one workgroup
// below takes it now);
// 3,000 ids, 7,000 power-law edges with 6.3M rows to the host 4.6 -> 1.6 ms (a
// round 5.6 us, the rest the copy; one wave per source had the hubs' rows to
// itself, up to 0.3 ms a round); 512 instances of 1,000 to 23,911 edges in
// one batch, the rounds alone 94 -> 11.7 ms.
#include "dlg_internal.h"

#include <algorithm>
#include <deque>

namespace dlg {

constexpr int TD_T = 256, TD_L = 16, TD_SUB = TD_T / TD_L;   // threads, lanes per task, tasks at a time
constexpr u32 TD_CW = 64;       // words per chunk (16 lanes x 4)
constexpr u32 TD_LONG = 256;    // predecessors above which a workgroup takes the row
constexpr u32 TD_LONG_WGS = 128;
constexpr int TD_SETS = 4;      // counter sets: a round's, the one before (published), the next (cleared)
constexpr int TD_SLOT = 8;      // words per counter slot: one 64-byte line
constexpr int TD_DEPTH = 4;     // rounds queued ahead of the host
static_assert(TD_DEPTH + 2 <= dlg_ctx::MAPPED_SLOTS, "every queued round has a mapped slot of its own");

// One id range (an instance): rows [row0, row0 + W), wpr words each (a
// multiple of 4) from word `base` (a whole emission tile), nc chunks per row,
// its first task and its first workgroup.
struct TdBlock {
    u64 base, task0;
    u32 row0, W, wpr, nc, wg0, pad;
};

struct TdArgs {
    const TdBlock *blk;
    const u32 *wgblk;        // the block of each task workgroup (null: one block)
    const u64 *off;          // predecessor lists by row
    const u32 *adj;          // predecessors as rows of their block
    const u32 *outdeg;       // out-degree (edges with their multiplicity) by row
    u32 *F;
    const uint2 *longs;      // (block, row) of the rows with long lists
    const u32 *nlong;
    unsigned long long *cnt; // TD_SETS sets of nslots slots: new tuples, their next join rows
    u32 *iters;              // per block: the first round without new tuples
    u32 *done;               // the round that published an empty one (0: none yet): later rounds do nothing
    u32 nslots, nblk, ntaskwg, per;   // task workgroups; tasks per sub-group
};

__device__ __forceinline__ u32 td_sub() { return threadIdx.x / TD_L; }
__device__ __forceinline__ bool td_any(const uint4 &v) { return (v.x | v.y | v.z | v.w) != 0u; }

// OR of the flagged predecessor chunks adj[p], p = first, first + 1 .. first +
// TD_L - 1, then `step` further on.  dc: the chunk column of D (this lane's
// four words of row 0), fc: its flag column.  Every lane of the wave calls it.
__device__ __forceinline__ uint4 td_gather(const u32 *adj, u64 first, u64 end, u64 step, const u32 *dc, u32 wpr,
                                           const unsigned char *fc, u32 nc, bool in_row) {
    const int l = threadIdx.x % TD_L, s0 = (threadIdx.x & (WAVE - 1)) & ~(TD_L - 1);
    uint4 acc = make_uint4(0u, 0u, 0u, 0u);
    for (u64 p = first; __ballot(p < end); p += step) {
        u32 z = 0;
        bool act = false;
        if (p + l < end) {
            z = adj[p + l];
            act = fc[(u64)z * nc] != 0;
        }
        u32 m = (u32)(__ballot(act) >> s0) & 0xffffu;   // this sub-group's flagged predecessors
        while (__ballot(m != 0u)) {
            uint4 v[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const bool has = m != 0u;
                const int j = has ? __ffs(m) - 1 : 0;
                m &= m - 1;   // 0 stays 0
                const u32 zz = (u32)__shfl((int)z, s0 + j, WAVE);
                v[k] = make_uint4(0u, 0u, 0u, 0u);
                if (has && in_row) v[k] = *(const uint4 *)(dc + (u64)zz * wpr);
            }
#pragma unroll
            for (int k = 0; k < 4; k++) {
                acc.x |= v[k].x;
                acc.y |= v[k].y;
                acc.z |= v[k].z;
                acc.w |= v[k].w;
            }
        }
    }
    return acc;
}

// The row's owner: acc & ~F into F and D (at `at`: this lane's words), the
// task's flag, and the new bits' count.  Every lane of the sub-group calls it.
__device__ __forceinline__ u32 td_update(uint4 acc, u32 *F, u32 *dn, u64 at, bool in_row, unsigned char *flag) {
    const int s0 = (threadIdx.x & (WAVE - 1)) & ~(TD_L - 1);
    uint4 n = make_uint4(0u, 0u, 0u, 0u);
    if (td_any(acc)) {   // lanes past the row hold none
        uint4 f = *(const uint4 *)(F + at);
        n = make_uint4(acc.x & ~f.x, acc.y & ~f.y, acc.z & ~f.z, acc.w & ~f.w);
        if (td_any(n)) {
            f = make_uint4(f.x | n.x, f.y | n.y, f.z | n.z, f.w | n.w);
            *(uint4 *)(F + at) = f;
        }
    }
    const bool has = ((u32)(__ballot(td_any(n)) >> s0) & 0xffffu) != 0u;
    if (has && in_row) *(uint4 *)(dn + at) = n;   // a flagged chunk is written whole
    if (threadIdx.x % TD_L == 0) *flag = has;
    return (u32)(__popc(n.x) + __popc(n.y) + __popc(n.z) + __popc(n.w));
}

// Whether round `round` has work.  Its own publisher may set `done` while it
// runs, which must not part a workgroup's waves: only earlier rounds' count.
__device__ __forceinline__ bool td_live(const TdArgs &a, u32 round) {
    const u32 d = *(volatile const u32 *)a.done;
    return d == 0u || d >= round;
}

// Round `round` (its predecessor's totals published first: those of round 0
// are the edges'), or only the publication (`publish_only`).
__global__ __launch_bounds__(TD_T) void td_round_k(TdArgs a, const u32 *dc, u32 *dn, const unsigned char *fc,
                                                   unsigned char *fn, u32 round, int publish_only, u64 *host, u64 seq) {
    __shared__ u64 s_c[TD_T / WAVE], s_w[TD_T / WAVE];
    __shared__ uint4 s_acc[TD_T];
    const int lane = threadIdx.x & (WAVE - 1), wv = threadIdx.x / WAVE, l = threadIdx.x % TD_L;
    u64 c = 0, w = 0;
    u32 slot = 0;
    const u32 set = round % TD_SETS;
    if (blockIdx.x == 0) {   // publishes the round before
        const unsigned long long *prev = a.cnt + (u64)((round - 1) % TD_SETS) * a.nslots * TD_SLOT;
        unsigned long long *next = a.cnt + (u64)((round + 1) % TD_SETS) * a.nslots * TD_SLOT;
        const bool was_done = *a.done != 0u;
        for (u32 i = threadIdx.x; i < a.nslots; i += TD_T) {
            const u64 v = prev[(u64)i * TD_SLOT];
            c += v;
            w += prev[(u64)i * TD_SLOT + 1];
            if (a.nblk > 1 && round > 1 && v == 0 && a.iters[i] == 0) a.iters[i] = round - 1;
            next[(u64)i * TD_SLOT] = 0;
            next[(u64)i * TD_SLOT + 1] = 0;
        }
        if (was_done) c = w = 0;
    } else if (td_live(a, round) && !publish_only) {
        const u32 wg = blockIdx.x - 1;
        if (wg < a.ntaskwg) {
            const u32 b = a.wgblk ? a.wgblk[wg] : 0u;
            const TdBlock k = a.blk[b];
            slot = a.nblk > 1 ? b : wg % a.nslots;
            const u64 ntask = (u64)k.W * k.nc;
            const u64 t0 = ((u64)(wg - k.wg0) * a.per) * TD_SUB + td_sub();
            for (u32 i = 0; i < a.per; i++) {
                const u64 t = t0 + (u64)i * TD_SUB;
                const bool valid = t < ntask;
                const u32 r = valid ? (u32)t / k.nc : 0u, ch = valid ? (u32)t - r * k.nc : 0u;
                const u64 p0 = a.off[k.row0 + r];
                u64 p1 = a.off[k.row0 + r + 1];
                const bool mine = valid && p1 - p0 <= (u64)TD_LONG;
                if (!mine) p1 = p0;
                const u32 col = ch * TD_CW + 4 * l;
                const bool in_row = col < k.wpr;
                const uint4 acc = td_gather(a.adj, p0, p1, TD_L, dc + k.base + col, k.wpr, fc + k.task0 + ch, k.nc, in_row);
                if (mine) {
                    const u32 n = td_update(acc, a.F, dn, k.base + (u64)r * k.wpr + col, in_row, fn + k.task0 + t);
                    c += n;
                    if (n) w += (u64)n * a.outdeg[k.row0 + r];
                }
            }
        } else {   // the rows with long lists: a workgroup per (row, chunk), its sub-groups' parts combined
            const u32 nl = *a.nlong;
            for (u32 i = wg - a.ntaskwg; i < nl; i += TD_LONG_WGS) {   // block-uniform
                const uint2 e = a.longs[i];
                const TdBlock k = a.blk[e.x];
                const u32 r = e.y;
                const u64 p0 = a.off[k.row0 + r], p1 = a.off[k.row0 + r + 1];
                u64 rc = 0;
                for (u32 ch = 0; ch < k.nc; ch++) {
                    const u32 col = ch * TD_CW + 4 * l;
                    const bool in_row = col < k.wpr;
                    uint4 acc = td_gather(a.adj, p0 + (u64)td_sub() * TD_L, p1, (u64)TD_SUB * TD_L, dc + k.base + col,
                                          k.wpr, fc + k.task0 + ch, k.nc, in_row);
                    s_acc[threadIdx.x] = acc;
                    __syncthreads();
                    if (td_sub() == 0) {
                        for (int s = 1; s < TD_SUB; s++) {
                            const uint4 v = s_acc[s * TD_L + l];
                            acc = make_uint4(acc.x | v.x, acc.y | v.y, acc.z | v.z, acc.w | v.w);
                        }
                        rc += td_update(acc, a.F, dn, k.base + (u64)r * k.wpr + col, in_row,
                                        fn + k.task0 + (u64)r * k.nc + ch);
                    }
                    __syncthreads();   // s_acc is rewritten for the next chunk
                }
                c += rc;
                if (rc) w += rc * a.outdeg[k.row0 + r];
                if (a.nblk > 1) {   // this row's block: its own slot
                    u64 x = rc;
#pragma unroll
                    for (int d = TD_L / 2; d > 0; d >>= 1) x += __shfl_xor(x, d, WAVE);
                    if (threadIdx.x == 0 && x)
                        atomicAdd(a.cnt + ((u64)set * a.nslots + e.x) * TD_SLOT, (unsigned long long)x);
                    c -= rc;
                }
            }
            slot = (wg - a.ntaskwg) % a.nslots;   // with several blocks only the join rows are left for it
        }
    }
#pragma unroll
    for (int d = WAVE / 2; d > 0; d >>= 1) {
        c += __shfl_xor(c, d, WAVE);
        w += __shfl_xor(w, d, WAVE);
    }
    if (lane == 0) {
        s_c[wv] = c;
        s_w[wv] = w;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    c = w = 0;
    for (int i = 0; i < TD_T / WAVE; i++) {
        c += s_c[i];
        w += s_w[i];
    }
    if (blockIdx.x == 0) {
        if (round > 1 && c == 0 && *a.done == 0u) *a.done = round;
        host[0] = c;
        host[1] = w;
        __threadfence_system();
        *(volatile u64 *)(host + dlg_ctx::MAPPED_SEQ) = seq;
        __threadfence_system();
        return;
    }
    unsigned long long *s = a.cnt + ((u64)set * a.nslots + slot) * TD_SLOT;
    if (c) atomicAdd(s, (unsigned long long)c);
    if (w) atomicAdd(s + 1, (unsigned long long)w);
}

// ---------------------------------------------------------------- set-up
__device__ __forceinline__ u32 td_key(int v, u32 lo) { return ((u32)v ^ 0x80000000u) - lo; }

__global__ void td_hist_k(const int2 *rows, u64 n, u32 lo, u32 *indeg, u32 *outdeg) {
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const int2 r = rows[i];
        atomicAdd(outdeg + td_key(r.x, lo), 1u);
        atomicAdd(indeg + td_key(r.y, lo), 1u);
    }
}

__device__ __forceinline__ u32 td_block_of(const TdBlock *blk, u32 nblk, u32 row) {
    u32 a = 0, b = nblk;   // the last block starting at or before the row
    while (b - a > 1) {
        const u32 m = (a + b) >> 1;
        if (blk[m].row0 <= row) a = m; else b = m;
    }
    return a;
}

// zero[0, zn), F[0, mn) and D[0, mn) cleared.
__global__ void td_clear_k(u64 *zero, u64 zn, uint4 *F, uint4 *D, u64 mn) {
    const u64 i0 = (u64)blockIdx.x * blockDim.x + threadIdx.x, stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = i0; i < mn; i += stride) F[i] = D[i] = make_uint4(0u, 0u, 0u, 0u);
    for (u64 i = i0; i < zn; i += stride) zero[i] = 0;
}

// The predecessor lists (indeg counts down to each list's next free place),
// the edges' bits in F and D with their tasks' flags, their distinct count and next join rows (slot
// of round 0), and the rows with long lists.
__global__ __launch_bounds__(TD_T) void td_fill_k(const int2 *rows, u64 n, u32 lo, u64 W, TdArgs a, u32 *indeg, u32 *adj,
                                                  u32 *D, unsigned char *flags, uint2 *longs, u32 *nlong) {
    __shared__ u64 s_c[TD_T / WAVE], s_w[TD_T / WAVE];
    u64 c = 0, w = 0;
    const u64 stride = (u64)gridDim.x * blockDim.x, t0 = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    for (u64 i = t0; i < n; i += stride) {
        const int2 e = rows[i];
        const u32 x = td_key(e.x, lo), z = td_key(e.y, lo);
        const TdBlock k = a.blk[a.nblk > 1 ? td_block_of(a.blk, a.nblk, z) : 0u];
        const u32 xr = x - k.row0, zr = z - k.row0;
        adj[a.off[z] + atomicSub(indeg + z, 1u) - 1u] = xr;
        const u64 at = k.base + (u64)zr * k.wpr + (xr >> 5);
        const u32 bit = 1u << (xr & 31);
        if (!(atomicOr(D + at, bit) & bit)) {
            atomicOr(a.F + at, bit);
            flags[k.task0 + (u64)zr * k.nc + (xr >> 5) / TD_CW] = 1;
            c++;
            w += a.outdeg[z];
        }
    }
    for (u64 r = t0; r < W; r += stride)
        if (a.off[r + 1] - a.off[r] > (u64)TD_LONG) {
            const u32 b = a.nblk > 1 ? td_block_of(a.blk, a.nblk, (u32)r) : 0u;
            longs[atomicAdd(nlong, 1u)] = make_uint2(b, (u32)r - a.blk[b].row0);
        }
#pragma unroll
    for (int d = WAVE / 2; d > 0; d >>= 1) {
        c += __shfl_xor(c, d, WAVE);
        w += __shfl_xor(w, d, WAVE);
    }
    if ((threadIdx.x & (WAVE - 1)) == 0) {
        s_c[threadIdx.x / WAVE] = c;
        s_w[threadIdx.x / WAVE] = w;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        c = w = 0;
        for (int i = 0; i < TD_T / WAVE; i++) {
            c += s_c[i];
            w += s_w[i];
        }
        unsigned long long *s = a.cnt + (u64)(blockIdx.x % a.nslots) * TD_SLOT;
        if (c) atomicAdd(s, (unsigned long long)c);
        if (w) atomicAdd(s + 1, (unsigned long long)w);
    }
}

__global__ void td_wgblk_k(const TdBlock *blk, u32 nblk, u32 nwg, u32 *wgblk) {
    const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nwg) return;
    u32 a = 0, b = nblk;
    while (b - a > 1) {
        const u32 m = (a + b) >> 1;
        if (blk[m].wg0 <= i) a = m; else b = m;
    }
    wgblk[i] = a;
}

// ---------------------------------------------------------- one workgroup's closure
// The whole run of a small range by one workgroup: F and D in LDS, the
// predecessors taken from the edges' own bits (row z of the first D holds z's predecessors),
// every round two barriers instead of a launch.  A thread keeps its words of N in
// registers while D is still read.  Takes what fits: 2 W wpr words, the out-degrees,
// the lists (2 bytes an edge): about 700 ids, less with many edges.
// Bound by the LDS reads of a round's predecessors and its two barriers.
constexpr int TS_T = 1024, TS_I = 5;              // threads, items (uint4s of the map) a thread at most
constexpr u32 TS_LONG = 128, TS_NLONG = 8;        // predecessors above which all threads share a row; such rows at most
constexpr u32 TS_LDS = 40000;                     // words: one workgroup's LDS but for 3.8 KB
constexpr u64 TS_MAX_ROWS = 8192;                 // edges, read by one workgroup

static u64 ts_words(u64 n, u64 W, u64 wpr) { return (2 * W + TS_NLONG) * wpr + 2 * W + 1 + (n + 1) / 2; }
static bool ts_takes(u64 n, u64 W, u64 wpr) {
    return n <= TS_MAX_ROWS && W <= (u64)TS_T && ts_words(n, W, wpr) <= TS_LDS && W * (wpr / 4) <= (u64)TS_T * TS_I;
}

__device__ __forceinline__ u64 ts_sum(u64 v, u64 *s_w) {   // every thread calls it; valid in thread 0
#pragma unroll
    for (int d = WAVE / 2; d > 0; d >>= 1) v += __shfl_xor(v, d, WAVE);
    if (threadIdx.x % WAVE == 0) s_w[threadIdx.x / WAVE] = v;
    __syncthreads();
    v = 0;
    if (threadIdx.x == 0)
        for (int w = 0; w < TS_T / WAVE; w++) v += s_w[w];
    __syncthreads();
    return v;
}

__global__ __launch_bounds__(TS_T) void td_small_k(const int2 *rows, u32 n, u32 lo, u32 W, u32 wpr, int max_it, u32 *out,
                                                   u32 out_words, u64 *host, u64 seq) {
    __shared__ __align__(16) u32 pool[TS_LDS];
    __shared__ u64 s_w[TS_T / WAVE + 1];
    __shared__ u32 s_long[TS_NLONG], s_nlong;
    const u32 mw = W * wpr, wq = wpr / 4, items = W * wq;
    u32 *D = pool, *F = pool + mw, *sums = F + mw, *outdeg = sums + TS_NLONG * wpr, *first = outdeg + W;   // first: W + 1 list starts
    unsigned short *adj = (unsigned short *)(first + W + 1);
    for (u32 i = threadIdx.x; i < mw; i += TS_T) D[i] = 0;
    if (threadIdx.x < W) outdeg[threadIdx.x] = 0;
    if (threadIdx.x == 0) s_nlong = 0;
    __syncthreads();
    for (u32 i = threadIdx.x; i < n; i += TS_T) {
        const int2 e = rows[i];
        const u32 x = td_key(e.x, lo), z = td_key(e.y, lo);
        atomicOr(D + z * wpr + (x >> 5), 1u << (x & 31));
        atomicAdd(outdeg + x, 1u);
    }
    __syncthreads();
    // the predecessors of row threadIdx.x, without duplicates; F = D
    u64 c = 0, w = 0;   // this thread's new tuples so far; the join rows that the last round's make
    {
        const u32 *row = D + threadIdx.x * wpr;
        u32 k = 0;
        if (threadIdx.x < W)
            for (u32 i = 0; i < wpr; i++) k += (u32)__popc(row[i]);
        u64 tot;
        u32 at = (u32)block_exclusive_scan<u64>((u64)k, s_w, &tot);
        if (threadIdx.x < W) {
            first[threadIdx.x] = at;
            if (threadIdx.x == W - 1) first[W] = (u32)tot;   // at most n
            for (u32 i = 0; i < wpr; i++)
                for (u32 b = row[i]; b; b &= b - 1) adj[at++] = (unsigned short)(i * 32 + (u32)__ffs(b) - 1);
            if (k > TS_LONG) {
                const u32 j = atomicAdd(&s_nlong, 1u);
                if (j < TS_NLONG) s_long[j] = threadIdx.x;
            }
            c = k;
            w = (u64)k * outdeg[threadIdx.x];
        }
    }
    uint4 *D4 = (uint4 *)D, *F4 = (uint4 *)F, *S4 = (uint4 *)sums;
    for (u32 i = threadIdx.x; i < items; i += TS_T) F4[i] = D4[i];
    u32 from[TS_I], to[TS_I], col[TS_I], deg[TS_I];
    __syncthreads();
    if (s_nlong > TS_NLONG) {   // block-uniform
        if (threadIdx.x == 0) {
            host[2] = 0;
            __threadfence_system();
            *(volatile u64 *)(host + dlg_ctx::MAPPED_SEQ) = seq;
            __threadfence_system();
        }
        return;
    }
#pragma unroll
    for (int q = 0; q < TS_I; q++) {
        const u32 i = threadIdx.x + (u32)q * TS_T, r = i < items ? i / wq : 0u;
        col[q] = i - r * wq;
        from[q] = i < items ? first[r] : 0u;
        to[q] = i < items ? first[r + 1] : 0u;   // past the end: an empty list
        deg[q] = outdeg[r];
        if (to[q] - from[q] > TS_LONG) to[q] = from[q];
    }
    const u32 nlong = s_nlong, part = TS_T / wq, slot = threadIdx.x / wq, scol = threadIdx.x % wq;
    int it = 0;
    u64 raw = 0;
    while (max_it <= 0 || it < max_it) {   // block-uniform; a round that finds nothing is the last, as F can only grow
        raw += w;
        w = 0;
        uint4 nw[TS_I];
        bool some = false;
        // the words of `a` that item i of F does not have, into F
        auto update = [&](uint4 a, u32 i, u32 dg) {
            const uint4 f = F4[i];
            a = make_uint4(a.x & ~f.x, a.y & ~f.y, a.z & ~f.z, a.w & ~f.w);
            if (td_any(a)) {
                F4[i] = make_uint4(f.x | a.x, f.y | a.y, f.z | a.z, f.w | a.w);
                const u32 k = (u32)(__popc(a.x) + __popc(a.y) + __popc(a.z) + __popc(a.w));
                c += k;
                w += (u64)k * dg;
                some = true;
            }
            return a;
        };
        if (nlong) {   // block-uniform
            for (u32 i = threadIdx.x; i < nlong * wq; i += TS_T) S4[i] = make_uint4(0u, 0u, 0u, 0u);
            __syncthreads();
            for (u32 j = 0; j < nlong; j++) {
                const u32 p1 = first[s_long[j] + 1];
                uint4 a = make_uint4(0u, 0u, 0u, 0u);
                if (slot < part)
                    for (u32 p = first[s_long[j]] + slot; p < p1; p += part) {
                        const uint4 v = D4[(u32)adj[p] * wq + scol];
                        a = make_uint4(a.x | v.x, a.y | v.y, a.z | v.z, a.w | v.w);
                    }
                u32 *sum = sums + (j * wq + scol) * 4;
                if (a.x) atomicOr(sum, a.x);
                if (a.y) atomicOr(sum + 1, a.y);
                if (a.z) atomicOr(sum + 2, a.z);
                if (a.w) atomicOr(sum + 3, a.w);
            }
            __syncthreads();
            for (u32 i = threadIdx.x; i < nlong * wq; i += TS_T) {
                const u32 r = s_long[i / wq];
                S4[i] = update(S4[i], r * wq + i % wq, outdeg[r]);
            }
        }
#pragma unroll
        for (int q = 0; q < TS_I; q++) {
            uint4 a = make_uint4(0u, 0u, 0u, 0u);
            for (u32 p = from[q]; p < to[q]; p += 4) {   // past the end the last one again
                uint4 v[4];
#pragma unroll
                for (int k = 0; k < 4; k++) v[k] = D4[(u32)adj[min(p + k, to[q] - 1)] * wq + col[q]];
#pragma unroll
                for (int k = 0; k < 4; k++) a = make_uint4(a.x | v[k].x, a.y | v[k].y, a.z | v[k].z, a.w | v[k].w);
            }
            if (td_any(a)) a = update(a, threadIdx.x + (u32)q * TS_T, deg[q]);
            nw[q] = a;
        }
        it++;
        const bool any = __syncthreads_or(some);   // D is read no more
        if (!any) break;
#pragma unroll
        for (int q = 0; q < TS_I; q++)
            if (threadIdx.x + (u32)q * TS_T < items) D4[threadIdx.x + (u32)q * TS_T] = nw[q];
        if (nlong) {
            __syncthreads();   // over the empty words that the rows' own threads have for them
            for (u32 i = threadIdx.x; i < nlong * wq; i += TS_T) D4[s_long[i / wq] * wq + i % wq] = S4[i];
        }
        __syncthreads();
    }
    for (u32 i = threadIdx.x; i < out_words / 4; i += TS_T) ((uint4 *)out)[i] = i < items ? F4[i] : make_uint4(0u, 0u, 0u, 0u);
    c = ts_sum(c, s_w);
    raw = ts_sum(raw, s_w);
    if (threadIdx.x == 0) {
        host[0] = c;
        host[1] = raw;
        host[2] = (u64)it;
        __threadfence_system();
        *(volatile u64 *)(host + dlg_ctx::MAPPED_SEQ) = seq;
        __threadfence_system();
    }
}

int tc_dense_run(dlg_ctx *ctx, const int32_t *d_rows, u64 n, u32 lo, u32 hi, const std::vector<u32> *starts, int max_it,
                 DBuf<u64> &out, u64 *total, u64 *raw, std::vector<int> *iters) {
    // the id ranges that hold rows, as in rowmap_init
    std::vector<u64> st;
    if (starts) st.assign(starts->begin(), starts->end());
    else st = {lo, (u64)hi + 1};
    if (st.back() == 0xffffffffull) st.back() = 0x100000000ull;   // a range that ends at the last id
    const u64 W = (u64)(hi - lo) + 1;
    std::vector<TdBlock> hb;
    std::vector<int> owner;   // the range each block is
    std::vector<MapRef> maps;
    // Tiles of 256 words where those of 2,048 would mostly pad (many instances of a few ids:
    // 100,000 of 10 took 2.4 GB of maps, and take 0.3): each map is there three times.
    u64 words = 0, tasks = 0, pad_big = 0, pad_small = 0;
    for (size_t i = 0; i + 1 < st.size(); i++) {
        const u64 b0 = std::max<u64>(st[i], lo), b1 = std::min<u64>(st[i + 1], (u64)hi + 1), w = b1 > b0 ? b1 - b0 : 0;
        pad_big += emit_tile_words(w * ((w + 127) / 128 * 4), false);
        pad_small += emit_tile_words(w * ((w + 127) / 128 * 4), true);
    }
    const bool small = 2 * pad_small <= pad_big;
    for (size_t i = 0; i + 1 < st.size(); i++) {
        const u64 b0 = std::max<u64>(st[i], lo), b1 = std::min<u64>(st[i + 1], (u64)hi + 1);
        if (b1 <= b0) continue;
        TdBlock k;
        k.W = (u32)(b1 - b0);
        k.wpr = (k.W + 127) / 128 * 4;
        k.nc = (k.wpr + TD_CW - 1) / TD_CW;
        k.row0 = (u32)(b0 - lo);
        k.base = words;
        k.task0 = tasks;
        k.wg0 = k.pad = 0;
        words += emit_tile_words((u64)k.W * k.wpr, small);
        tasks += (u64)k.W * k.nc;
        hb.push_back(k);
        owner.push_back((int)i);
        maps.push_back({(u32)b0, k.W, k.wpr, k.base});
    }
    if (!starts && ts_takes(n, W, hb[0].wpr)) {
        DBuf<u32> F(ctx, words);
        const u64 seq = ++ctx->mapped_seq;
        DLG_LAUNCH(ctx, DLG_K_BITMAP_INSERT, 8.0 * n + 4.0 * words, td_small_k, 1, TS_T, 0, (const int2 *)d_rows, (u32)n, lo,
                   (u32)W, hb[0].wpr, max_it, F.p, (u32)words, ctx->mapped_dev(seq), seq);
        ctx->wait_mapped(seq);
        const volatile u64 *m = ctx->mapped_host(seq);
        const int it = (int)m[2];
        if (it > 0) {   // 0: too many rows with long lists
            *total = m[0];
            *raw += m[1];
            bitmap_emit_tiled(ctx, F.p, maps, words, out, *total, small);
            if (iters) iters->assign(1, it);
            return it;
        }
    }
    const u32 nblk = (u32)hb.size();
    // four tasks per sub-group once that still leaves every CU eight workgroups
    const u32 per = tasks >= (u64)ctx->num_cus * 8 * TD_SUB * 4 ? 4u : 1u;
    u64 nwg = 0;
    for (TdBlock &k : hb) {
        k.wg0 = (u32)nwg;
        nwg += ((u64)k.W * k.nc + per * TD_SUB - 1) / (per * TD_SUB);
    }
    if (nwg + TD_LONG_WGS + 1 > 0x7fffffffull) fail(DLG_OVERFLOW, "TC maps: too many tasks");
    TdArgs a;
    a.nblk = nblk;
    a.nslots = nblk > 1 ? nblk : 64u;
    a.ntaskwg = (u32)nwg;
    a.per = per;
    // one block of cleared words: degrees (in: W, out: W), flags of D, counters, long-row count, done, iterations
    const u64 fw = (tasks + 7) / 8;   // flags in u64s
    const u64 cw = (u64)TD_SETS * a.nslots * TD_SLOT;
    const u64 zw = fw + cw + (2 * W + nblk + 3) / 2;
    DBuf<u64> zero(ctx, zw);
    unsigned char *flags = (unsigned char *)zero.p;
    a.cnt = (unsigned long long *)(zero.p + fw);
    u32 *z32 = (u32 *)(zero.p + fw + cw);
    u32 *indeg = z32, *outdeg = z32 + W;
    a.iters = outdeg + W;
    u32 *nlong = a.iters + nblk;
    a.done = nlong + 1;
    a.nlong = nlong;
    a.outdeg = outdeg;
    DBuf<u32> F(ctx, words), D2(ctx, 2 * words);   // D twice: a round reads one and writes the other
    DBuf<u64> flags2(ctx, fw ? fw : 1), off(ctx, W + 1), tab(ctx, sizeof(TdBlock) / 8 * nblk);
    DBuf<u32> adj(ctx, n), wgblk(ctx);
    DBuf<uint2> longs(ctx, n / TD_LONG + 1);
    a.F = F.p;
    u32 *D[2] = {D2.p, D2.p + words};
    unsigned char *fl[2] = {flags, (unsigned char *)flags2.p};
    a.blk = (const TdBlock *)tab.p;
    a.off = off.p;
    a.adj = adj.p;
    a.longs = longs.p;
    HIPCHK(hipMemcpyAsync(tab.p, hb.data(), sizeof(TdBlock) * nblk, hipMemcpyHostToDevice, ctx->stream));
    DLG_LAUNCH(ctx, DLG_K_MISC, 8.0 * (zw + words), td_clear_k, sgrid(ctx, std::max(zw, words / 4)), ctx->block_size, 0, zero.p, zw,
               (uint4 *)F.p, (uint4 *)D[0], words / 4);
    a.wgblk = nullptr;
    if (nblk > 1) {
        wgblk.ensure(nwg);
        DLG_LAUNCH(ctx, DLG_K_MISC, 4.0 * nwg, td_wgblk_k, grid_for(nwg, 256), 256, 0, a.blk, nblk, (u32)nwg, wgblk.p);
        a.wgblk = wgblk.p;
    }
    DLG_LAUNCH(ctx, DLG_K_MISC, 16.0 * n, td_hist_k, sgrid(ctx, n), ctx->block_size, 0, (const int2 *)d_rows, n, lo,
               indeg, outdeg);
    scan_u32_u64_async(ctx, indeg, W, off.p, off.p + W);
    const unsigned fg = (unsigned)std::min<u64>((std::max(n, W) + TD_T - 1) / TD_T, (u64)ctx->num_cus * 8);
    DLG_LAUNCH(ctx, DLG_K_MISC, 40.0 * n, td_fill_k, fg, TD_T, 0, (const int2 *)d_rows, n, lo, W, a, indeg, adj.p, D[0],
               fl[0], longs.p, nlong);
    // The rounds, up to TD_DEPTH queued ahead of the host.  Kernel r publishes
    // round r - 1 (round 0: the edges); a round that found nothing lets the
    // queued ones do nothing.
    const unsigned g = (unsigned)nwg + TD_LONG_WGS + 1;
    std::deque<u64> q;   // sequence numbers of the rounds not read yet, from round `it` on
    u32 launched = 0;
    auto launch = [&](bool publish_only) {
        const u32 r = launched + 1;
        const u64 seq = ++ctx->mapped_seq;
        DLG_LAUNCH(ctx, DLG_K_BITMAP_INSERT, 0.0, td_round_k, publish_only ? 1u : g, TD_T, 0, a, (const u32 *)D[(r - 1) & 1],
                   D[r & 1], (const unsigned char *)fl[(r - 1) & 1], fl[r & 1], r, publish_only ? 1 : 0,
                   ctx->mapped_dev(seq), seq);
        if (!publish_only) launched++;
        q.push_back(seq);
    };
    int it = -1;   // rounds read; round 0 is the edges
    u64 rows_next = 0;
    *total = 0;
    while (true) {
        while ((int)launched < it + 2 + TD_DEPTH && (max_it <= 0 || (int)launched < max_it)) launch(false);
        if (q.empty()) launch(true);   // the last round asked for
        const u64 seq = q.front();
        q.pop_front();
        ctx->wait_mapped(seq);
        const volatile u64 *m = ctx->mapped_host(seq);
        const u64 nn = m[0], w = m[1];
        it++;
        *total += nn;
        if (it > 0) *raw += rows_next;   // the rows this round joined
        rows_next = w;
        // algorithmic bytes of a round: its rows' words that changed cannot be known without
        // counting them; the new tuples' bits read and written are what is left
        ctx->prof_add_bytes(DLG_K_BITMAP_INSERT, nn / 4.0);
        if (it > 0 && (nn == 0 || (max_it > 0 && it >= max_it))) break;
    }
    if (iters) {
        std::vector<u32> h(nblk);
        if (nblk > 1) {
            HIPCHK(hipMemcpyAsync(h.data(), a.iters, 4 * nblk, hipMemcpyDeviceToHost, ctx->stream));
            ctx->sync();
        }
        iters->assign(st.size() - 1, 1);   // a range without rows finds nothing in round one
        for (u32 b = 0; b < nblk; b++) (*iters)[owner[b]] = nblk > 1 && h[b] ? (int)h[b] : it;
    }
    D2.release();   // before the relation itself is allocated
    bitmap_emit_tiled(ctx, a.F, maps, words, out, *total, small);
    return it;
}

}  // namespace dlg
