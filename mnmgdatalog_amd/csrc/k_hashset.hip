// k_hashset.hip -- device hash set of tuples: the full relation of wide id ranges.
//
// unique(J) \ F and F u N (tc.cu:250-283) in one step: every join row goes
// into the set as it is formed, and the rows that claim a slot are the new
// tuples, appended to the relation's array.  J is never written or sorted.
// Slots are u64 tuples, linear probing from a 64-bit
// mix of the tuple, EMPTY = all ones; the one tuple equal to EMPTY
// ((INT32_MAX, INT32_MAX)) is kept in a flag instead of a slot.
#include "dlg_internal.h"

#include <algorithm>
#include <deque>
#include <cmath>
#include <type_traits>

namespace dlg {

__device__ __forceinline__ u64 mix64(u64 x) {
    // SplitMix64 finaliser (Steele, Lea, Flood 2014)
    x ^= x >> 30;
    x *= 0xbf58476d1ce4e5b9ull;
    x ^= x >> 27;
    x *= 0x94d049bb133111ebull;
    x ^= x >> 31;
    return x;
}

// Insert tuples known to be absent and pairwise distinct.
__global__ void hs_insert_k(const u64 *x, u64 n, u64 *slots, u64 mask, u32 *flag) {
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    u64 stride = (u64)gridDim.x * blockDim.x;
    for (; i < n; i += stride) {
        u64 v = x[i];
        if (v == EMPTY_SLOT) {
            *flag = 1u;
            continue;
        }
        u64 p = mix64(v) & mask;
        while (true) {
            unsigned long long prev = atomicCAS((unsigned long long *)&slots[p],
                                                (unsigned long long)EMPTY_SLOT, (unsigned long long)v);
            if (prev == EMPTY_SLOT) break;
            p = (p + 1) & mask;
        }
    }
}

void hashset_reserve(dlg_ctx *ctx, HashSet &hs, u64 need, double lf, const u64 *all, u64 n_all) {
    if (!(lf > 0.0)) lf = ctx->load_factor;
    lf = std::min(0.9, std::max(0.1, lf));
    if (hs.cap && (double)need <= lf * (double)hs.cap) return;
    u64 want = (u64)std::ceil((double)need / lf);
    u64 cap = hs.cap ? hs.cap : 1024;
    while (cap < want || cap <= need) cap <<= 1;
    hs.cap = 0;   // no table, should there be no memory for the new one
    hs.slots.ensure(cap);
    hs.cap = cap;
    if (!hs.flag.p) hs.flag.ensure(1);
    fill_u64(ctx, hs.slots.p, cap, EMPTY_SLOT);
    fill_u32(ctx, hs.flag.p, 1, 0u);
    hs.count = 0;
    if (n_all) hashset_insert(ctx, hs, all, n_all);   // rehash what the set already held
}

void hashset_insert(dlg_ctx *ctx, HashSet &hs, const u64 *x, u64 n) {
    if (!n) return;
    // a tuple read, one slot line and a CAS per element
    DLG_LAUNCH(ctx, DLG_K_HSET_INSERT, 24.0 * n, hs_insert_k, sgrid(ctx, n), ctx->block_size, 0, x, n,
               hs.slots.p, hs.cap - 1, hs.flag.p);
    hs.count += n;
}

// ---------------------------------------------------------------- insertion of join rows
__device__ __forceinline__ u64 hs_cas(u64 *slot, u64 t) {
    return atomicCAS((unsigned long long *)slot, (unsigned long long)EMPTY_SLOT, (unsigned long long)t);
}

// True when t was absent: a slot from p on is claimed for it (t's slots
// before p hold other tuples).  A plain read first: a slot never changes once
// set, and a stale empty one only costs the CAS.
__device__ __forceinline__ bool hs_claim(u64 *slots, u64 mask, u64 t, u64 p) {
    while (true) {
        u64 s = slots[p];
        if (s == EMPTY_SLOT) {
            s = hs_cas(&slots[p], t);
            if (s == EMPTY_SLOT) return true;
        }
        if (s == t) return false;
        p = (p + 1) & mask;
    }
}

// A tile's rows t[] (valid: ok[]) into the set; the new ones appended at
// all[*count ..], one counter atomic per tile.  Bound by the latency of the
// slot reads and CASes: a thread's I first slots are read together, then
// claimed together where they are empty, and only rows whose first slot
// holds another tuple go on one by one.  Tiles of one row per thread keep
// small rounds (tens of thousands of rows) on every CU: 54,000 rows a round
// 16 us against 53 us by tiles of 8 rows per thread, claimed one by one (TC of
// 400,000 ids, 68 rounds: 4.1 against 6.5 ms, and 16.5 ms when the join was
// written, sorted and looked up).
constexpr int HJ_T = 256;
constexpr int HJ_BIG = 8;                    // rows per thread of the large rounds
constexpr u64 HJ_BIG_MIN = 1ull << 19;       // probes from which tiles of HJ_BIG rows per thread fill the chip

template <int I>
__device__ __forceinline__ void hs_insert_tile(const u64 (&t)[I], const bool (&ok)[I], u64 *slots, u64 mask, u32 *flag,
                                               u64 *all, unsigned long long *count, u64 *sc, u64 *s_base) {
    u64 pos[I], s[I];
    bool real[I];   // a row whose tuple has a slot of its own
#pragma unroll
    for (int r = 0; r < I; r++) {
        real[r] = ok[r] && t[r] != EMPTY_SLOT;
        pos[r] = mix64(t[r]) & mask;
        s[r] = real[r] ? slots[pos[r]] : 0ull;
    }
    u64 got[I];
#pragma unroll
    for (int r = 0; r < I; r++) got[r] = real[r] && s[r] == EMPTY_SLOT ? hs_cas(&slots[pos[r]], t[r]) : s[r];
    u32 fresh = 0;
#pragma unroll
    for (int r = 0; r < I; r++) {
        if (!real[r]) {
            if (ok[r] && atomicExch(flag, 1u) == 0u) fresh |= 1u << r;
            continue;
        }
        if (got[r] == EMPTY_SLOT || (got[r] != t[r] && hs_claim(slots, mask, t[r], (pos[r] + 1) & mask))) fresh |= 1u << r;
    }
    u64 tot;
    u64 o = block_exclusive_scan<u64>((u64)__popc(fresh), sc, &tot);
    if (threadIdx.x == 0) *s_base = tot ? atomicAdd(count, (unsigned long long)tot) : 0ull;
    __syncthreads();
    o += *s_base;
#pragma unroll
    for (int r = 0; r < I; r++)
        if ((fresh >> r) & 1u) all[o++] = t[r];
}

// The join rows [r0, min(*total, r0 + room)) of a counted join (its probes'
// row starts and offsets) into the set: persistent workgroups over tiles of
// HJ_TILE rows, a tile's probes staged in LDS as in join_expand_k.
// NODIAG drops the rows with key == value.
template <int PROJ, bool NODIAG, int HJ_I>
__global__ __launch_bounds__(HJ_T) void hs_join_insert_k(const u64 *probe, u64 np, const u32 *pstart, const u64 *offs,
                                                         u64 r0, u64 room, const u64 *rows, u64 *slots, u64 mask,
                                                         u32 *flag, u64 *all, unsigned long long *count) {
    constexpr int HJ_TILE = HJ_T * HJ_I;
    constexpr u32 HJ_STAGE = HJ_TILE + 1;   // probes of a tile staged in LDS (a probe with rows adds at least one)
    __shared__ u64 s_lo, s_hi, s_base;
    __shared__ u64 sc[HJ_T / WAVE + 1];
    __shared__ u32 l_offs[HJ_STAGE], l_start[HJ_STAGE], l_pv[HJ_STAGE];
    const u64 all_rows = offs[np], end = all_rows < r0 + room ? all_rows : r0 + room;
    for (u64 base = r0 + (u64)blockIdx.x * HJ_TILE; base < end; base += (u64)gridDim.x * HJ_TILE) {   // block-uniform
        if (threadIdx.x < WAVE) {   // the first wave finds the tile's probes
            const u64 last = (base + HJ_TILE < end ? base + HJ_TILE : end) - 1;
            const u64 lo = wave_upper_bound(offs, 0, np, base) - 1;
            const u64 hi = wave_upper_bound(offs, lo, np, last);
            if (threadIdx.x == 0) {
                s_lo = lo;
                s_hi = hi;
            }
        }
        __syncthreads();
        const u64 lo = s_lo, span = s_hi - lo;
        const bool staged = span <= (u64)HJ_STAGE;
        if (staged)
            for (u64 j = threadIdx.x; j < span; j += HJ_T) {
                u64 of = offs[lo + j];
                u32 st = pstart[lo + j];
                if (j == 0) {   // the tile may start inside the first probe's rows
                    st += (u32)(base - of);
                    of = base;
                }
                l_offs[j] = (u32)(of - base);
                l_start[j] = st;
                l_pv[j] = tval(probe[lo + j]);
            }
        __syncthreads();
        u64 t[HJ_I];
        bool ok[HJ_I];
        u32 idx[HJ_I], pv[HJ_I];
#pragma unroll
        for (int r = 0; r < HJ_I; r++) {
            const u64 o = base + (u64)r * HJ_T + threadIdx.x;
            ok[r] = o < end;
            idx[r] = pv[r] = 0;
            if (!ok[r]) continue;
            if (staged) {
                const u32 rel = (u32)(o - base);
                u32 a = 0, b = (u32)span;   // the last probe starting at or before the row
                while (b - a > 1) {
                    const u32 m = (a + b) >> 1;
                    if (l_offs[m] <= rel) a = m; else b = m;
                }
                idx[r] = l_start[a] + (rel - l_offs[a]);
                pv[r] = l_pv[a];
            } else {   // a tile spanning more probes (runs of probes without rows)
                const u64 i = upper_bound_u64(offs, lo, lo + span, o) - 1;
                idx[r] = pstart[i] + (u32)(o - offs[i]);
                pv[r] = tval(probe[i]);
            }
        }
        u32 hv[HJ_I];
#pragma unroll
        for (int r = 0; r < HJ_I; r++) hv[r] = ok[r] ? tval(rows[idx[r]]) : 0u;
#pragma unroll
        for (int r = 0; r < HJ_I; r++) {
            t[r] = PROJ == DLG_PROJ_HV_PV ? tmake(hv[r], pv[r]) : tmake(pv[r], hv[r]);
            if (NODIAG) ok[r] = ok[r] && hv[r] != pv[r];
        }
        hs_insert_tile(t, ok, slots, mask, flag, all, count, sc, &s_base);
        __syncthreads();   // the staging is rewritten for the next tile
    }
}

template <int HJ_I>
__global__ __launch_bounds__(HJ_T) void hs_list_insert_k(const u64 *x, u64 n, u64 *slots, u64 mask, u32 *flag, u64 *all,
                                                         unsigned long long *count) {
    constexpr int HJ_TILE = HJ_T * HJ_I;
    __shared__ u64 s_base;
    __shared__ u64 sc[HJ_T / WAVE + 1];
    for (u64 base = (u64)blockIdx.x * HJ_TILE; base < n; base += (u64)gridDim.x * HJ_TILE) {   // block-uniform
        u64 t[HJ_I];
        bool ok[HJ_I];
#pragma unroll
        for (int r = 0; r < HJ_I; r++) {
            const u64 i = base + (u64)r * HJ_T + threadIdx.x;
            ok[r] = i < n;
            t[r] = ok[r] ? x[i] : 0ull;
        }
        hs_insert_tile(t, ok, slots, mask, flag, all, count, sc, &s_base);
        __syncthreads();   // s_base and sc are rewritten by the next tile
    }
}

// The relation's size and the join's rows (offs + np, or null) to the host.
__global__ void hs_publish_k(const u64 *count, const u64 *rows, u64 *host, u64 seq) {
    if (threadIdx.x != 0) return;
    host[0] = *count;
    host[1] = rows ? *rows : 0ull;
    __threadfence_system();
    *(volatile u64 *)(host + dlg_ctx::MAPPED_SEQ) = seq;
    __threadfence_system();
}

static void hs_publish(dlg_ctx *ctx, const u64 *count, const u64 *rows, u64 *h) {
    const u64 seq = ++ctx->mapped_seq;
    DLG_LAUNCH(ctx, DLG_K_MISC, 0.0, hs_publish_k, 1, 64, 0, count, rows, ctx->mapped_dev(seq), seq);
    ctx->wait_mapped(seq);
    const volatile u64 *m = ctx->mapped_host(seq);
    h[0] = m[0];
    h[1] = m[1];
}

// Room for `want` more tuples: the table and the array grow together (the
// array holds every tuple the table may, lf of its slots), to twice the relation at least:
// by what is asked for alone, TC of 400,000 ids took 2 % longer for filling tables anew.
// Short of memory they grow by that, and the slots are filled further first.
constexpr double HS_TIGHT_LF = 0.8;
constexpr u64 HS_LEAST = 1ull << 16, HS_LARGE = 1ull << 24;
static void hs_grow(dlg_ctx *ctx, HashRel &r, u64 want) {
    const u64 need = r.n + want;
    if (r.hs.cap && need <= r.limit) return;
    const double lf = r.tight ? std::max(r.lf, HS_TIGHT_LF) : r.lf;
    hashset_reserve(ctx, r.hs, r.tight ? need : std::max(need, 2 * r.n), lf, r.all.p, r.n);
    u64 limit = std::max(need, (u64)(lf * (double)r.hs.cap));
    if (r.all.cap < limit) {
        DBuf<u64> g(ctx);
        try {
            g.ensure(limit);
        } catch (const Error &e) {   // what is asked for, then
            if (e.status != DLG_OUT_OF_MEMORY) throw;
            limit = need;
            if (r.all.cap < limit) g.ensure(limit);
        }
        if (g.p) {
            copy_u64(ctx, g.p, r.all.p, r.n);
            r.all = std::move(g);
        }
    }
    r.limit = limit;
    if (!r.count.p) {
        r.count.ensure(1);
        fill_u64(ctx, r.count.p, 1, 0ull);
    }
}

// No memory for what was asked for: from here on as little as will do.
static void hs_short(HashRel &r, const Error &e) {
    if (e.status != DLG_OUT_OF_MEMORY) throw e;
    r.tight = true;
    r.hs.slots.release();
    r.hs.cap = 0;
}

// The same, or, short of memory, room for HS_LEAST of them.
static void hs_grow_some(dlg_ctx *ctx, HashRel &r, u64 want) {
    const u64 had = r.limit - r.n, least = std::min(want, HS_LEAST);
    if (!r.tight) {
        try {
            return hs_grow(ctx, r, want);
        } catch (const Error &e) {
            hs_short(r, e);
        }
    }
    if (!r.hs.cap || had < least) hs_grow(ctx, r, std::max(had, least));
}

static unsigned hs_grid(const dlg_ctx *ctx, u64 rows, u64 tile) {
    return (unsigned)std::max<u64>(1, std::min<u64>((rows + tile - 1) / tile, (u64)ctx->num_cus * 8));
}

u64 hashrel_insert_list(dlg_ctx *ctx, HashRel &r, const u64 *x, u64 n) {
    if (n == 0) return 0;
    hs_grow(ctx, r, n);
    auto go = [&](auto kern, int per) {
        DLG_LAUNCH(ctx, DLG_K_HSET_INSERT, 24.0 * n, kern, hs_grid(ctx, n, (u64)HJ_T * per), HJ_T, 0, x, n, r.hs.slots.p,
                   r.hs.cap - 1, r.hs.flag.p, r.all.p, (unsigned long long *)r.count.p);
    };
    if (n >= HJ_BIG_MIN) go(hs_list_insert_k<HJ_BIG>, HJ_BIG);
    else go(hs_list_insert_k<1>, 1);
    u64 h[2];
    hs_publish(ctx, r.count.p, nullptr, h);
    const u64 nn = h[0] - r.n;
    r.n = h[0];
    return nn;
}

u64 hashrel_insert_join(dlg_ctx *ctx, HashRel &r, const Index &ix, const u64 *probe, u64 off, u64 n, int proj,
                        bool nodiag, JoinScratch &js, u64 *raw) {
    if (n == 0 || ix.n == 0) return 0;
    const u64 before = r.n;
    join_count_async(ctx, ix, probe ? probe : r.all.p + off, n, js);
    // room for about what the rows will be; the rows past it wait for more.  A set that takes a
    // millisecond to fill anew is used as it is first: after a hub's round the rows are many and
    // hardly any new (below that, room ahead of the next rounds is worth more: TC of 930,000 random
    // edges 6.4 ms, 6.8 without)
    const bool some = r.n >= HS_LARGE && r.hs.cap && r.limit - r.n >= n / 2;
    if (!some) hs_grow_some(ctx, r, 2 * n);
    u64 r0 = 0;
    while (true) {
        const u64 room = r.limit - r.n;
        const u64 *pr = probe ? probe : r.all.p + off;   // growing moves the array
        auto go = [&](auto kern, int per) {
            DLG_LAUNCH(ctx, DLG_K_HSET_INSERT, 24.0 * n, kern, hs_grid(ctx, room, (u64)HJ_T * per), HJ_T, 0, pr, n,
                       (const u32 *)js.pstart.p, (const u64 *)js.offs.p, r0, room, (const u64 *)ix.rows.p, r.hs.slots.p,
                       r.hs.cap - 1, r.hs.flag.p, r.all.p, (unsigned long long *)r.count.p);
        };
        auto sized = [&](auto proj_c, auto nodiag_c) {
            if (n >= HJ_BIG_MIN) go(hs_join_insert_k<proj_c.value, nodiag_c.value, HJ_BIG>, HJ_BIG);
            else go(hs_join_insert_k<proj_c.value, nodiag_c.value, 1>, 1);
        };
        using std::integral_constant;
        if (proj == DLG_PROJ_PV_HV) {
            if (nodiag) sized(integral_constant<int, DLG_PROJ_PV_HV>(), std::true_type());
            else sized(integral_constant<int, DLG_PROJ_PV_HV>(), std::false_type());
        } else {
            if (nodiag) sized(integral_constant<int, DLG_PROJ_HV_PV>(), std::true_type());
            else sized(integral_constant<int, DLG_PROJ_HV_PV>(), std::false_type());
        }
        u64 h[2];
        hs_publish(ctx, r.count.p, js.offs.p + n, h);
        const u64 fresh = h[0] - r.n;
        r.n = h[0];
        if (r0 == 0) *raw += h[1];
        r0 += room;
        if (r0 >= h[1]) break;
        // as long as most rows are new, room for eight times the relation, as the table is filled
        // anew each time it grows: a star's 38M pairs from 15,000 edges 14.0 ms by doubling, 9.8 so and
        // 6.9 with the rule above; SG's 400M from 20,000 97 and 59 (77 by sorting the rows)
        const u64 left = h[1] - r0;
        hs_grow_some(ctx, r, std::min(left, std::max<u64>(2 * fresh >= room ? std::max(8 * r.n, 2 * n) : r.n, 1ull << 20)));
    }
    return r.n - before;
}

// ------------------------------------------------- rounds queued ahead of the host
// A TC round over wide ids in one launch: a workgroup takes HJ_T probes, finds
// their runs in the index, lays the runs end to end by a block scan and inserts
// the rows, so the counts and offsets of a whole round are never written or scanned; and
// a round reads its place from the state that the rounds before left, so HR_DEPTH
// of them are queued ahead of the host (kernel r publishes round r - 1's totals).
// A round that would fill the table past its limit, or whose tile of probes has
// more than HR_ROWS rows (a hub, which one workgroup would take alone), stalls: the rounds
// behind it do nothing, and the host runs it again by hashrel_insert_join, which
// finds what it had appended in the set.
// Bound by the latency of its chain: probe, slot, run, row, set slot, append.  With
// a count, a scan of up to three launches, an insertion, a publication and a wait for
// the host in every round: TC of 400,000 ids and 360,000 random edges (69 rounds)
// 3.4 -> 1.9 ms; of 1,000,000 and 930,000 (115) 7.0 -> 4.9; a path of 3,000 (a round
// 27 -> 12.6 us) 82 -> 38; 3,000 power-law ids in a wide range 3.9 -> 3.5.
constexpr int HR_DEPTH = 3, HR_SETS = 4;
constexpr u64 HR_ROWS = 1ull << 14;
// Room that rounds queued ahead may ask for beyond the relation: what the largest of them
// take when every row is new, or a quarter of the relation.  The room is counted in join rows,
// as a tile cannot know which of its own are new; a round of many more rows than new tuples
// (cliques) runs by itself, which asks for room as its tuples come: 700 ids with 40,000 edges
// held 840 MB for 490,000 tuples, and hold 82 so (2.0 -> 2.2 ms).
constexpr u64 HR_ROOM = 2 * (HR_DEPTH + 1) * HJ_BIG_MIN;
static_assert(HR_DEPTH + 2 <= dlg_ctx::MAPPED_SLOTS, "every queued round has a mapped slot of its own");

struct HrState {
    unsigned long long end[HR_SETS];     // by round % HR_SETS: the relation before the round
    unsigned long long fresh[HR_SETS];   // the round's new tuples
    unsigned long long used[HR_SETS];    // its join rows
    u32 stall, skew;                     // the round that stalled (0: none); that a tile of it has too many rows
};

// Round 0: what the first round finds as Δ.
__global__ void hr_init_k(HrState *st, u64 off, u64 n) {
    const u32 i = threadIdx.x;
    if (i < HR_SETS) {
        st->end[i] = i ? 0ull : off;
        st->fresh[i] = i ? 0ull : n;
        st->used[i] = 0ull;
    }
    if (i == 0) st->stall = st->skew = 0u;
}

__global__ __launch_bounds__(HJ_T) void hr_round_k(HrState *st, u32 round, int publish_only, u64 limit, const u64 *ix_slots,
                                                   u64 ix_mask, const u32 *gstart, const u64 *rows, u64 *slots, u64 mask,
                                                   u32 *flag, u64 *all, u64 *host, u64 seq) {
    __shared__ u64 sc[HJ_T / WAVE + 1], s_base, l_offs[HJ_T];
    __shared__ u32 l_start[HJ_T], l_pv[HJ_T];
    __shared__ bool s_ok;
    const u32 prev = (round - 1) % HR_SETS, cur = round % HR_SETS, next = (round + 1) % HR_SETS;
    const u64 beg = st->end[prev], np = st->fresh[prev], end = beg + np;   // left by earlier launches
    // an earlier round's stall only: this round may set it while its workgroups read it
    const u32 stall = *(volatile const u32 *)&st->stall;
    const bool is_void = stall != 0u && stall < round;
    if (blockIdx.x == 0) {   // publishes the round before
        if (threadIdx.x != 0) return;
        st->end[cur] = end;
        st->fresh[next] = st->used[next] = 0ull;
        host[0] = end;
        host[1] = st->used[prev];
        host[2] = is_void ? 1u + (st->skew != 0u) : 0u;
        __threadfence_system();
        *(volatile u64 *)(host + dlg_ctx::MAPPED_SEQ) = seq;
        __threadfence_system();
        return;
    }
    if (is_void || publish_only) return;
    for (u64 tile = (u64)(blockIdx.x - 1) * HJ_T; tile < np; tile += (u64)(gridDim.x - 1) * HJ_T) {   // block-uniform
        const u64 i = tile + threadIdx.x;
        u32 c = 0, s = 0, pv = 0;
        if (i < np) {
            const u64 t = all[beg + i];
            pv = tval(t);
            const u32 g = ix_find(ix_slots, ix_mask, tkey(t));
            if (g != 0xffffffffu) {
                s = gstart[g];
                c = gstart[g + 1] - s;
            }
        }
        u64 tot;
        l_offs[threadIdx.x] = block_exclusive_scan<u64>((u64)c, sc, &tot);
        l_start[threadIdx.x] = s;
        l_pv[threadIdx.x] = pv;
        if (threadIdx.x == 0) {
            const u64 u = tot ? atomicAdd(&st->used[cur], (unsigned long long)tot) : 0ull;
            s_ok = tot <= HR_ROWS && end + u + tot <= limit;
            if (!s_ok) {
                if (tot > HR_ROWS) st->skew = 1u;
                st->stall = round;
            }
        }
        __syncthreads();
        if (!s_ok) return;   // block-uniform
        for (u64 base = 0; base < tot; base += HJ_T) {
            const u64 o = base + threadIdx.x;
            const bool ok[1] = {o < tot};
            u32 a = 0, b = HJ_T;   // the last probe whose run starts at or before the row
            while (b - a > 1) {
                const u32 m = (a + b) >> 1;
                if (l_offs[m] <= o) a = m; else b = m;
            }
            const u64 t[1] = {ok[0] ? tmake(tval(rows[(u64)l_start[a] + (o - l_offs[a])]), l_pv[a]) : 0ull};
            hs_insert_tile<1>(t, ok, slots, mask, flag, all + end, &st->fresh[cur], sc, &s_base);
            __syncthreads();   // s_base and sc are rewritten
        }
        __syncthreads();   // and the staging
    }
}

int hashrel_rounds(dlg_ctx *ctx, HashRel &r, const Index &ix, u64 off, u64 n, int max_it, JoinScratch &js, u64 *raw) {
    const bool slots = n != 0 && ix.n != 0 && !ix.sorted && ix.dense_w == 0 && ix.nslots != 0;
    DBuf<u64> state(ctx, (sizeof(HrState) + 7) / 8);
    HrState *st = (HrState *)state.p;
    bool plain = !slots;   // rounds one by one
    int it = 0, stalls = 0;
    u64 per = n;   // what a round may need room for: the last one's rows
    // a round by itself, `known` tuples before it; false: the last
    auto alone = [&](u64 known) {
        u64 rows = 0;
        hashrel_insert_join(ctx, r, ix, nullptr, off, n, DLG_PROJ_HV_PV, false, js, &rows);
        *raw += rows;
        it++;
        off += n;
        n = r.n - known;
        per = std::max(n, rows);
        return n != 0 && !(max_it > 0 && it >= max_it);
    };
    while (true) {
        const u64 ahead = 2 * (HR_DEPTH + 1) * per;
        if (plain || n >= HJ_BIG_MIN || ahead > std::max(HR_ROOM, r.n / 4)) {   // large rounds have threads of several rows each
            if (!alone(r.n)) return it;
            continue;
        }
        try {
            hs_grow(ctx, r, ahead);
        } catch (const Error &e) {   // no memory for so many rounds at once
            hs_short(r, e);
            plain = true;
            continue;
        }
        DLG_LAUNCH(ctx, DLG_K_MISC, 0.0, hr_init_k, 1, 64, 0, st, off, n);
        std::deque<u64> q;            // sequence numbers of the publications not read yet
        u32 launched = 0, pub = 0;    // rounds launched; whose totals are read next
        const int it0 = it;
        bool closing = false;         // no more rounds of this stretch
        auto launch = [&](bool publish_only) {
            const u64 seq = ++ctx->mapped_seq;
            // workgroups for twice the probes of the last round known
            const unsigned g = publish_only ? 1u : 1u + hs_grid(ctx, std::min<u64>(2 * n, (u64)ctx->num_cus * 4 * HJ_T), HJ_T);
            DLG_LAUNCH(ctx, DLG_K_HSET_INSERT, 24.0 * n, hr_round_k, g, HJ_T, 0, st, launched + 1, publish_only ? 1 : 0, r.limit,
                       (const u64 *)ix.slots.p, ix.nslots - 1, (const u32 *)ix.gstart.p, (const u64 *)ix.rows.p, r.hs.slots.p,
                       r.hs.cap - 1, r.hs.flag.p, r.all.p, ctx->mapped_dev(seq), seq);
            if (!publish_only) launched++;
            q.push_back(seq);
        };
        while (true) {
            while (!closing && launched < pub + HR_DEPTH && (max_it <= 0 || it0 + (int)launched < max_it)) launch(false);
            if (q.empty()) launch(true);   // nothing behind the last round publishes it
            const u64 seq = q.front();
            q.pop_front();
            ctx->wait_mapped(seq);
            const volatile u64 *m = ctx->mapped_host(seq);
            const u64 end = m[0], rows = m[1], stall = m[2];
            if (pub++ == 0) continue;   // Δ itself
            r.n = end;
            if (stall) {
                ctx->sync();   // the rounds behind it have passed without work
                fill_u64(ctx, r.count.p, 1, r.n);
                if (pub > 4) stalls = 0;
                plain = stall == 2 || ++stalls > 2;
                if (!alone(off + n)) return it;
                break;
            }
            *raw += rows;
            it++;
            off += n;
            n = end - off;
            const bool last = n == 0 || (max_it > 0 && it >= max_it);
            per = std::max(n, rows);
            closing = closing || n >= HJ_BIG_MIN || r.limit - r.n < (HR_DEPTH + 1) * per;   // the rounds launched may take as much each
            if (!last && !(closing && pub > launched)) continue;
            fill_u64(ctx, r.count.p, 1, r.n);
            if (last) return it;
            break;
        }
    }
}

}  // namespace dlg
