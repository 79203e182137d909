// k_tcrings.hip -- TC rounds over exactly symmetric graphs of small degree, as
// lists of words.
//
// Let S_r(x) be the ends that a TC round r finds for the source x (those of the
// shortest walks of r + 1 edges).  A round is
//     S_r+1(x) = (union of S_r(y) over the neighbours y of x) \ everything before,
// and in a symmetric graph a neighbour of an end at walk length l has length
// l - 1, l or l + 1 (it is one step from that end, and that end from it), so
// "everything before" is S_r(x) and S_r-1(x): the rounds need nothing of the full
// relation F, whose words a round otherwise reads and writes one by one (a 64-byte
// line each way for 2.6 new bits).  Rings of a graph in a locality order are few
// bits in few words, so S_r(x) is a list of (word, bits).
//
//   tc_ring_k   a wave takes 8 sources; for each, a bitmap row in LDS takes the
//               neighbours' lists (OR), loses its own last two (AND NOT), and
//               gives the rest up word by word (exchange with 0, which also
//               leaves it empty) as the new list
//   tc_ring_merge_k   F row by row in LDS: the lists of all rounds of the buffers
//               ORed in at once, when they are full and at the end
// Lists live in two buffers that are filled in turn, one round after another, a
// region per 1/512 of the workgroups (one counter each: device atomics on one
// line serialise).  The host turns from one to the other when it sees the end
// coming, and merges both when both are full (a row read and written once for
// dozens of rounds).  A round that finds a region full all the same marks itself
// void, and is launched again in the other buffer.  A buffer holds two rounds at
// least, so the lists that the next round reads are never in the one being filled
// anew; the buffers begin with half of F's bytes each and grow fourfold, to room
// for two rounds of any size, while few rounds fill them.  Rounds are queued ahead
// of the host (round r publishes r - 1's totals).
//
// Bound by the latency of a source's chain (its lists, then three LDS steps) at the
// 8 waves per CU that a 20 KB bitmap row leaves: 5,400 cycles a source and round.
// All rows of a round ran 480 us with the loads in turn, 258 with a row's all in
// flight, 214 with the parts below dealt to the XCDs instead of eighths, and 181
// with steps of up to 1,024 entries, no branch per step, and the reservation
// behind the first row's loads.  Persistent waves that read a source ahead: 250.
//
// Whole calls against the row kernel (k_tcrows.hip): the 400 x 400 grid (edges
// kept at 0.55, 1 % shortcuts; 540 rounds, 2.07e10 tuples) 450 -> 220 ms, of which
// the rounds 353 -> 100 and the merges 27; the whole 200 x 200 grid 48 -> 23; a
// symmetric road network of 129,000 ids (617 rounds) 354 -> 145; 600 rounds of a
// path of 20,000 ids 32 -> 14; a binary tree of 131,000 ids 257 -> 48; random graphs
// of degree 6 and 40,000 ids 53 -> 17; 130 x 130 18 -> 10; sparse rests (cycles of 2
// and 10, a grid kept at 0.45) 1.0 to 1.05 times as fast.
#include "dlg_internal.h"

#include <algorithm>
#include <deque>
#include <type_traits>

namespace dlg {

constexpr u32 TG_EMPTY = 0xffffffffu;
constexpr int TG_D = 8, TG_R = WAVE / TG_D;   // neighbours per source (a lane each), sources per wave
constexpr u32 TG_XCD = 8, TG_PARTS = 64, TG_REGIONS = 512, TG_SLOTS = 64;
constexpr int TG_SETS = 4, TG_LINE = 8;
constexpr int TG_DEPTH = 4;                   // rounds queued ahead of the host
constexpr u32 TG_META = 64;                   // rounds per buffer at most
constexpr int TG_MT = 256;                    // threads of the merge
constexpr u32 TG_SPARSE = 32;                 // rows with fewer entries than 1 / 32 of their words are merged word by word
static_assert(TG_DEPTH + 2 <= dlg_ctx::MAPPED_SLOTS, "every queued round has a mapped slot of its own");

// A round's lists: S(x) is words[pos[x] ..][0, len[x]).
struct TgLists {
    u32 *pos, *len;
    uint2 *words;
};
struct TgArgs {
    const u32 *ell;            // TG_D neighbours per source, TG_EMPTY past its degree
    const u32 *deg;            // out degrees, edges counted as often as they are given
    u32 W, wpr;
    unsigned long long *bump;  // a region's entries in use, a line each
    u64 region;                // entries per region
    unsigned long long *cnt;   // TG_SETS sets of TG_SLOTS lines: new tuples, the next round's join rows, entries moved
    u32 *done, *full;          // the round that published an empty one; the round that found a region full (0: none); full = done + 1
    u32 *live;                 // a workgroup's sources: the last round that gave a neighbour of theirs a list
};

__device__ __forceinline__ void tg_fence() {   // a wave's LDS operations stay in order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ u64 tg_sum(u64 v) {
#pragma unroll
    for (int d = WAVE / 2; d > 0; d >>= 1) v += __shfl_xor(v, d, WAVE);
    return v;
}
__device__ __forceinline__ u32 tg_rank(u64 bal) {
    return __builtin_amdgcn_mbcnt_hi((u32)(bal >> 32), __builtin_amdgcn_mbcnt_lo((u32)bal, 0u));
}
__device__ __forceinline__ u32 tg_lane(u32 v, int lane) { return (u32)__builtin_amdgcn_readlane((int)v, lane); }

// What a launch of the round kernel does: the round and the publication of the
// last one's totals, only that, or only the round (launched again: the host has
// the last one's totals, which later rounds may have cleared).
enum { TG_BOTH = 0, TG_PUBLISH = 1, TG_ROUND = 2 };

// Publishes round `round` - 1 and clears the next set.
__device__ __forceinline__ void tg_publish(const TgArgs &a, u32 round, int mode, u64 *host, u64 seq) {
    static_assert(TG_SLOTS == WAVE, "a line per lane");
    unsigned long long *prev = a.cnt + ((u64)((round - 1) % TG_SETS) * TG_SLOTS + threadIdx.x) * TG_LINE;
    unsigned long long *next = a.cnt + ((u64)((round + 1) % TG_SETS) * TG_SLOTS + threadIdx.x) * TG_LINE;
    u64 t[3], use = 0;
#pragma unroll
    for (int q = 0; q < 3; q++) {
        t[q] = tg_sum(prev[q]);
        next[q] = 0;
    }
    for (u32 i = threadIdx.x; i < TG_REGIONS; i += WAVE) use = max(use, (u64)a.bump[(u64)i * TG_LINE]);
#pragma unroll
    for (int d = WAVE / 2; d > 0; d >>= 1) use = max(use, (u64)__shfl_xor(use, d, WAVE));
    if (threadIdx.x == 0 && mode != TG_ROUND) {
        const u32 f = *(volatile const u32 *)a.full;   // set by an earlier round: it and those after it are void
        const bool is_void = f != 0 && f < round;
        if (!is_void && round > 1 && t[0] == 0 && *a.done == 0u) *a.done = round;
        for (int q = 0; q < 3; q++) host[q] = t[q];
        host[3] = is_void;
        host[4] = use;   // the fullest region's entries (this round may have begun to reserve)
        __threadfence_system();
        *(volatile u64 *)(host + dlg_ctx::MAPPED_SEQ) = seq;
        __threadfence_system();
    }
}

__device__ __forceinline__ void tg_count(const TgArgs &a, u32 round, u32 slot, u64 nn, u64 raw, u64 moved) {
    nn = tg_sum(nn);
    raw = tg_sum(raw);
    if (threadIdx.x == 0) {
        unsigned long long *c = a.cnt + ((u64)(round % TG_SETS) * TG_SLOTS + slot % TG_SLOTS) * TG_LINE;
        if (nn) atomicAdd(c, (unsigned long long)nn);
        if (raw) atomicAdd(c + 1, (unsigned long long)raw);
        if (moved) atomicAdd(c + 2, (unsigned long long)moved);
    }
}

// Where a source's entries are, for its wave: T of up to NL neighbours, list k at
// `last` + q[k] from the concatenation's entry p[k] on; O of its own last two.
template <int NL>
struct TgRow {
    u32 T, L1, O;
    const uint2 *w1, *w0;
    u32 p[NL], q[NL];
    __device__ __forceinline__ TgRow(int l0, u32 t, u32 pre, u32 np, u32 ol, u32 op, const uint2 *last, const uint2 *prev) {
        T = t;
        L1 = tg_lane(ol, l0);
        O = L1 + tg_lane(ol, l0 + 1);
        w1 = last + tg_lane(op, l0);
        w0 = O > L1 ? prev + tg_lane(op, l0 + 1) - L1 : w1;
#pragma unroll
        for (int k = 0; k < NL; k++) {
            p[k] = tg_lane(pre, l0 + k);
            q[k] = tg_lane(np, l0 + k) - p[k];
        }
    }
    // Entries c + lane, c + 64 + lane, ... (a lane past the end reads the last again)
    template <int NS>
    __device__ __forceinline__ void load(uint2 (&e)[NS], u32 c, const uint2 *last) const {
        u32 o[NS];
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const u32 t = min(c + s * WAVE + threadIdx.x, T - 1);
            o[s] = q[0];
#pragma unroll
            for (int k = 1; k < NL; k++) o[s] = t >= p[k] ? q[k] : o[s];
            o[s] += t;
        }
#pragma unroll
        for (int s = 0; s < NS; s++) e[s] = last[o[s]];
    }
    template <int NS>
    __device__ __forceinline__ void own(uint2 (&f)[NS], u32 c) const {
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const u32 t = min(c + s * WAVE + threadIdx.x, max(O, 1u) - 1);
            f[s] = (t < L1 ? w1 : w0)[t];
        }
    }
};

// The steps of a row on what has been read: the neighbours' words in, the own
// ones out, the rest to words[cur ..] (cur moved on, its bits added).  A lane
// past the end works on a word of its own behind the map (`pad`), with no bits.
template <int NS>
__device__ __forceinline__ void tg_in(u32 *map, uint2 (&e)[NS], u32 c, u32 T, u32 pad) {
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const bool in = c + s * WAVE + threadIdx.x < T;
        e[s].x = in ? e[s].x : pad;
        atomicOr(map + e[s].x, in ? e[s].y : 0u);
    }
}
template <int NS>
__device__ __forceinline__ void tg_out(u32 *map, const uint2 (&f)[NS], u32 c, u32 O, u32 pad) {
#pragma unroll
    for (int s = 0; s < NS; s++) atomicAnd(map + (c + s * WAVE + threadIdx.x < O ? f[s].x : pad), ~f[s].y);
}
template <int NS>
__device__ __forceinline__ void tg_take(u32 *map, const uint2 (&e)[NS], uint2 *words, u32 &cur, u32 &bits) {
    u32 v[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) v[s] = atomicExch(map + e[s].x, 0u);   // a word's first taker has it
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const u64 bal = __ballot(v[s] != 0u);
        if (v[s]) words[cur + tg_rank(bal)] = make_uint2(e[s].x, v[s]);
        cur += (u32)__popcll(bal);
        bits += (u32)__popc(v[s]);
    }
}

// Round `round` (its lists to `out`) from the last round's lists and those of
// the one before, the last round's totals published first.
__global__ __launch_bounds__(WAVE, 4) void tc_ring_k(TgArgs a, TgLists last, TgLists prev, TgLists out, u32 round,
                                                  int mode, u64 *host, u64 seq) {
    extern __shared__ uint4 tg_map4[];
    u32 *map = (u32 *)tg_map4;
    if (blockIdx.x == 0) {
        tg_publish(a, round, mode, host, seq);
        return;
    }
    const u64 state = *(volatile const u64 *)a.done;   // one wave: no waves to part
    const u32 stop = (u32)state, full = (u32)(state >> 32);
    if (mode == TG_PUBLISH || (full && full < round)) return;
    // The sources go to the XCDs (workgroup b to XCD b % 8) in 64 parts in turn: near sources share an L2, and an
    // XCD has parts from everywhere, as the rings' sizes differ along the order.
    const u32 b = blockIdx.x - 1, nb = (a.W + TG_R - 1) / TG_R, part = (nb + TG_PARTS - 1) / TG_PARTS;
    const u32 turn = b / TG_XCD / part, blk = (turn * TG_XCD + b % TG_XCD) * part + (b / TG_XCD - turn * part);
    if (blk >= nb) return;
    const u32 slot = b % TG_REGIONS;
    const int lane = threadIdx.x, j = lane % TG_D, r = lane / TG_D;
    const u32 x = blk * TG_R + (u32)r;
    if ((stop && stop < round) || a.live[blk] + 1 < round) {   // nothing left, or nothing near: empty lists
        if (j == 0 && x < a.W) out.pos[x] = out.len[x] = 0;
        return;
    }
    // lane 8 r + j: neighbour j of source r, its list; lanes 8 r and 8 r + 1 also the source's own two
    const u32 id = x < a.W ? a.ell[(u64)x * TG_D + j] : TG_EMPTY;
    u32 np = 0, nl = 0, op = 0, ol = 0, dg = 0;
    if (x < a.W) {
        dg = a.deg[x];
        if (j < 2) {
            ol = j ? prev.len[x] : last.len[x];
            op = j ? prev.pos[x] : last.pos[x];
        }
    }
    if (id != TG_EMPTY) {
        nl = last.len[id];
        np = last.pos[id];
    }
    u32 inc = nl;
#pragma unroll
    for (int d = 1; d < TG_D; d <<= 1) {
        const u32 t = (u32)__shfl_up((int)inc, d, TG_D);
        if (j >= d) inc += t;
    }
    const u32 pre = inc - nl;
    const u32 need = (u32)tg_sum(j == TG_D - 1 ? min(inc, a.wpr) : 0u);   // a list has a word once
    u32 olen = 0, opos = 0;
    u64 nn = 0, raw = 0, moved = 0;
    if (need) {
        u64 at = 0;
        if (lane == 0) at = atomicAdd(a.bump + (u64)slot * TG_LINE, (unsigned long long)need);   // used from the first source's end on
        const u32 own = ol + (u32)__shfl_xor((int)ol, 1, WAVE);   // in lanes 8 r, 8 r + 1
        const u32 pad = (a.wpr + 3) / 4 * 4 + lane;
        for (u32 i = lane; i < (a.wpr + 3) / 4 + WAVE / 4; i += WAVE) tg_map4[i] = make_uint4(0u, 0u, 0u, 0u);
        tg_fence();
        u64 todo = __ballot(j == TG_D - 1 && inc != 0u);   // bit 8 r + 7: source r has candidates
        u32 cur = 0, start = 0;
        bool placed = false;
        while (todo) {   // wave-uniform
            const int l0 = __ffsll((unsigned long long)todo) - TG_D;
            todo &= todo - 1;
            const u32 T = tg_lane(inc, l0 + TG_D - 1), O = tg_lane(own, l0), most = max(T, O);
            const bool few = tg_lane(pre, l0 + TG_D / 2) == T;   // no entries past the fourth neighbour
            u32 bits = 0, from = 0;
            // where the lists go, once: false if the region is full
            auto place = [&]() {
                if (!placed) {
                    at = __shfl(at, 0, WAVE);
                    if (at + need > a.region) return false;
                    cur = start = (u32)(slot * a.region + at);
                    placed = true;
                }
                from = cur;
                return true;
            };
            // all of the row's entries read at once
            auto whole = [&](auto steps) {
                constexpr int NS = decltype(steps)::value;
                const TgRow<TG_D / 2> row(l0, T, pre, np, ol, op, last.words, prev.words);
                uint2 e[NS], f[NS];
                row.load(e, 0, last.words);
                row.own(f, 0);
                tg_in(map, e, 0, T, pad);
                tg_fence();
                tg_out(map, f, 0, O, pad);
                tg_fence();
                if (!place()) return false;
                tg_take(map, e, out.words, cur, bits);
                tg_fence();
                return true;
            };
            bool ok;
            if (few && most <= 4 * WAVE) ok = whole(std::integral_constant<int, 4>());
            else if (few && most <= 8 * WAVE) ok = whole(std::integral_constant<int, 8>());
            else if (few && most <= 16 * WAVE) ok = whole(std::integral_constant<int, 16>());
            else {   // 512 at a time, the neighbours' twice
                constexpr u32 C = 8 * WAVE;
                const TgRow<TG_D> row(l0, T, pre, np, ol, op, last.words, prev.words);
                uint2 e[8];
                for (u32 c = 0; c < T; c += C) {
                    row.load(e, c, last.words);
                    tg_in(map, e, c, T, pad);
                }
                tg_fence();
                for (u32 c = 0; c < O; c += C) {
                    row.own(e, c);
                    tg_out(map, e, c, O, pad);
                }
                tg_fence();
                ok = place();
                for (u32 c = 0; ok && c < T; c += C) {
                    row.load(e, c, last.words);
#pragma unroll
                    for (int s = 0; s < 8; s++)
                        if (c + s * WAVE + lane >= T) e[s].x = pad;
                    tg_take(map, e, out.words, cur, bits);
                }
                tg_fence();
            }
            if (!ok) {
                if (lane == 0) *a.full = round;
                return;
            }
            if (r == l0 / TG_D) {   // in all eight of its lanes
                opos = from;
                olen = cur - from;
            }
            nn += bits;
            raw += (u64)bits * tg_lane(dg, l0);
            moved += T + O + (cur - from);
        }
        // what was not used goes back, unless another wave has reserved since
        if (lane == 0 && cur - start < need)
            atomicCAS(a.bump + (u64)slot * TG_LINE, (unsigned long long)(at + need), (unsigned long long)(at + (cur - start)));
    }
    if (j == 0 && x < a.W) {
        out.pos[x] = opos;
        out.len[x] = olen;
    }
    if (olen && id != TG_EMPTY) a.live[id / TG_R] = round;   // symmetric: its neighbours' next candidates
    tg_count(a, round, slot, nn, raw, moved);
}

// Round 0's lists, the neighbours themselves, and empty ones before them.
__global__ __launch_bounds__(WAVE) void tc_ring_init_k(TgArgs a, TgLists out, u32 *none) {
    const int lane = threadIdx.x, j = lane % TG_D, r = lane / TG_D;
    const u32 x = blockIdx.x * TG_R + (u32)r, slot = blockIdx.x % TG_REGIONS;
    const u32 id = x < a.W ? a.ell[(u64)x * TG_D + j] : TG_EMPTY;
    const u32 w = id == TG_EMPTY ? TG_EMPTY : id >> 5;
    u32 v = id == TG_EMPTY ? 0u : 1u << (id & 31);
    bool head = v != 0;   // the word's first lane of the source
    const u32 own = v;
#pragma unroll
    for (int d = 1; d < TG_D; d++) {
        const int o = (j + d) % TG_D;
        const u32 w2 = (u32)__shfl((int)w, lane - j + o, WAVE), v2 = (u32)__shfl((int)own, lane - j + o, WAVE);
        if (w2 == w && own) {
            v |= v2;
            if (o < j) head = false;
        }
    }
    const u64 bal = __ballot(head);
    u64 at = 0;
    if (lane == 0) at = atomicAdd(a.bump + (u64)slot * TG_LINE, (unsigned long long)__popcll(bal));
    at = slot * a.region + __shfl(at, 0, WAVE);
    if (head) out.words[at + tg_rank(bal)] = make_uint2(w, v);
    const u64 mine = (bal >> (lane - j)) & 0xffull;
    if (j == 0 && x < a.W) {
        out.pos[x] = (u32)at + (u32)__popcll(bal & ((1ull << lane) - 1ull));
        out.len[x] = (u32)__popcll(mine);
        none[x] = 0;
    }
    const u32 c = head ? (u32)__popc(v) : 0u;
    tg_count(a, 0, slot, c, c ? (u64)c * a.deg[x] : 0, 0);
}

// F's row x (in LDS) takes its lists of the first k[i] rounds of buffer i.
struct TgMerge {
    const u32 *pos[2], *len[2];
    const uint2 *words[2];
    u32 k[2];
};
__global__ __launch_bounds__(TG_MT) void tc_ring_merge_k(u32 *F, u32 wpr, u32 W, TgMerge g) {
    extern __shared__ uint4 tg_map4[];
    u32 *map = (u32 *)tg_map4;
    __shared__ u32 s_pos[2 * TG_META], s_len[2 * TG_META];
    static_assert(2 * TG_META <= TG_MT, "a thread per round");
    const u32 x = blockIdx.x, k0 = g.k[0], k = k0 + g.k[1];
    u32 n = 0;
    if (threadIdx.x < k) {
        const u32 i = threadIdx.x < k0 ? 0u : 1u, m = threadIdx.x - (i ? k0 : 0u);
        s_pos[threadIdx.x] = g.pos[i][(u64)m * W + x];
        s_len[threadIdx.x] = n = g.len[i][(u64)m * W + x];
    }
    u32 *row = F + (u64)x * wpr;
    const u32 lane = threadIdx.x & (WAVE - 1);
    __shared__ u32 s_all;
    if (threadIdx.x == 0) s_all = 0;
    __syncthreads();
    if (n) atomicAdd(&s_all, n);
    __syncthreads();
    if (s_all * TG_SPARSE < wpr) {   // block-uniform: word by word (two rounds may share one) instead of the whole row
        for (u32 m = threadIdx.x / WAVE; m < k; m += TG_MT / WAVE)
            for (u32 i = lane; i < s_len[m]; i += WAVE) {
                const uint2 e = g.words[m < k0 ? 0 : 1][s_pos[m] + i];
                atomicOr(row + e.x, e.y);
            }
        return;
    }
    for (u32 i = threadIdx.x; i < wpr; i += TG_MT) map[i] = row[i];
    __syncthreads();
    for (u32 m = threadIdx.x / WAVE; m < k; m += TG_MT / WAVE) {
        const u32 L = s_len[m];
        const uint2 *w = g.words[m < k0 ? 0 : 1] + s_pos[m];
        for (u32 i = 0; i < L; i += 4 * WAVE) {   // a lane past the end takes the last entry again
            uint2 e[4];
#pragma unroll
            for (u32 s = 0; s < 4; s++) e[s] = w[min(i + s * WAVE + lane, L - 1)];
#pragma unroll
            for (u32 s = 0; s < 4; s++)
                if (i + s * WAVE + lane < L) atomicOr(map + e[s].x, e[s].y);
        }
    }
    __syncthreads();
    for (u32 i = threadIdx.x; i < wpr; i += TG_MT) row[i] = map[i];
}

// The buffers turned: regions empty, no round void, the counters of `round` cleared.
__global__ __launch_bounds__(WAVE) void tc_ring_turn_k(TgArgs a, u32 round) {
    for (u32 i = threadIdx.x; i < TG_REGIONS; i += WAVE) a.bump[(u64)i * TG_LINE] = 0;
    unsigned long long *c = a.cnt + ((u64)(round % TG_SETS) * TG_SLOTS + threadIdx.x) * TG_LINE;
    c[0] = c[1] = c[2] = 0;
    if (threadIdx.x == 0) *a.full = 0;
}

// Entries per region at most: two rounds of any size, as a workgroup's sources have at most every word each.
static constexpr u64 tg_region_max(u64 W, u64 wpr) {
    const u64 grid = TG_PARTS * (((W + TG_R - 1) / TG_R + TG_PARTS - 1) / TG_PARTS);
    return 2 * ((grid + TG_REGIONS - 1) / TG_REGIONS) * TG_R * wpr;
}

// Rows of which seven fit a CU's LDS (184,320 ids).  Wider ones leave too few waves for the
// chain that a round is: parts of paths, 4,500 to 7,200 rounds, against the row kernel 370 and
// 427 ms at 160,000 ids, 431 and 435 at 180,000, 604 and 568 at 200,000, 1,169 and 776 at 262,016;
// grids of 8,100 ids each 68 and 84, 84 and 98, 98 and 110, 160 and 147.
constexpr u64 TG_MAX_WPR = 5760;
static_assert(TG_REGIONS * tg_region_max(32 * TG_MAX_WPR, TG_MAX_WPR) < 1ull << 32, "list positions are 32-bit");

bool tc_rings_takes(const TcRows &tr, const RowMap &F) {
    if (!tr.ell.p || F.blocks.size() != 1) return false;
    const u64 wpr = F.blocks[0].wpr;
    return wpr >= TG_D && wpr <= TG_MAX_WPR;
}

// One run with buffers of region[i] entries per region to begin with; -1 (F then
// holds part of the result) if a buffer turns out not to hold two rounds.
static int tg_run(dlg_ctx *ctx, const TcRows &tr, RowMap &F, int max_it, u64 first_region, u64 *total, u64 *raw) {
    const u64 W = F.W, wpr = F.blocks[0].wpr, nb = (W + TG_R - 1) / TG_R, grid = TG_PARTS * ((nb + TG_PARTS - 1) / TG_PARTS);
    TgArgs a;
    a.ell = tr.ell.p;
    a.deg = tr.deg.p;
    a.W = (u32)W;
    a.wpr = (u32)wpr;
    const u64 region_max = tg_region_max(W, wpr);
    u64 region[2] = {first_region, first_region};
    const u64 cw = (u64)TG_SETS * TG_SLOTS * TG_LINE, bw = (u64)TG_REGIONS * TG_LINE;
    DBuf<u64> state(ctx, cw + bw + 1 + (nb + 1) / 2);
    DBuf<uint2> words[2] = {DBuf<uint2>(ctx, TG_REGIONS * region[0]), DBuf<uint2>(ctx, TG_REGIONS * region[1])};
    DBuf<u32> pos[2] = {DBuf<u32>(ctx, TG_META * W), DBuf<u32>(ctx, TG_META * W)};
    DBuf<u32> len[2] = {DBuf<u32>(ctx, TG_META * W), DBuf<u32>(ctx, TG_META * W)};
    fill_u64(ctx, state.p, cw + bw + 1 + (nb + 1) / 2, 0ull);   // `live` too: every source is round 0's
    a.cnt = (unsigned long long *)state.p;
    a.bump = (unsigned long long *)state.p + cw;
    a.done = (u32 *)(state.p + cw + bw);
    a.full = a.done + 1;
    a.live = a.full + 1;
    a.region = region[0];
    const unsigned lds = (unsigned)((wpr + 3) / 4 * 16);   // a row; the rounds also have a word per lane behind it
    auto lists = [&](int buf, u32 m) { return TgLists{pos[buf].p + (u64)m * W, len[buf].p + (u64)m * W, words[buf].p}; };
    // the buffer being filled, its rounds so far; the last two rounds' lists (round 0's, and none before it)
    int buf = 0;
    u32 used = 1;
    struct Round {
        int buf;
        u32 m, held;   // its place; the other buffer's rounds that are not merged yet
    };
    u32 held = 0;
    std::deque<Round> at;   // the rounds from `it` - 1 on that were launched
    DLG_LAUNCH(ctx, DLG_K_MISC, 40.0 * W, tc_ring_init_k, (unsigned)nb, WAVE, 0, a, lists(0, 0), lists(1, TG_META - 1).len);
    at.push_back({1, TG_META - 1, 0});   // round -1: its lengths are all 0
    at.push_back({0, 0, 0});
    // the first k lists of the buffer being filled and the other's held ones into F
    auto merge = [&](u32 k) {
        TgMerge g;
        for (int i = 0; i < 2; i++) {
            const int bf = i ? buf : buf ^ 1;
            g.pos[i] = pos[bf].p;
            g.len[i] = len[bf].p;
            g.words[i] = words[bf].p;
            g.k[i] = i ? k : held;
        }
        if (g.k[0] + g.k[1])
            DLG_LAUNCH(ctx, DLG_K_BITMAP_INSERT, 8.0 * F.nwords, tc_ring_merge_k, (unsigned)W, TG_MT, lds, F.words.p, a.wpr, a.W,
                       g);
        held = 0;
    };
    // round `next` starts the other buffer (all rounds before it are known), whose lists and this one's `rounds` are merged first if it still has some
    auto turn = [&](u32 rounds, u32 next) {
        if (held) merge(rounds);
        else held = rounds;
        buf ^= 1;
        used = 0;
        // filled by few rounds: the next one larger (it holds nothing that is still needed)
        if (rounds < TG_META / 2 && region[buf] <= region[buf ^ 1] && region[buf] < region_max) {
            const u64 more = std::min(4 * region[buf ^ 1], region_max);
            words[buf].release();
            try {
                words[buf].ensure(TG_REGIONS * more);
                region[buf] = more;
            } catch (const Error &e) {
                if (e.status != DLG_OUT_OF_MEMORY) throw;
                words[buf].ensure(TG_REGIONS * region[buf]);
            }
        }
        a.region = region[buf];
        DLG_LAUNCH(ctx, DLG_K_MISC, 0.0, tc_ring_turn_k, 1, WAVE, 0, a, next);
    };
    std::deque<u64> q;   // sequence numbers of the rounds not read yet, from round `it` + 1 on
    int launched = 0, it = -1;
    u64 use = 0, growth = 0;   // the fullest region's entries after the last round known, and what a round may add
    int use_buf = 0;           // in this buffer
    auto launch = [&](int mode) {
        const u32 r = (u32)launched + 1;
        const u64 seq = mode != TG_ROUND ? ++ctx->mapped_seq : 0;
        const Round p1 = at.back(), p0 = at[at.size() - 2];
        DLG_LAUNCH(ctx, DLG_K_BITMAP_INSERT, 0.0, tc_ring_k, mode == TG_PUBLISH ? 1u : 1u + (unsigned)grid, WAVE, lds + 4 * WAVE, a,
                   lists(p1.buf, p1.m), lists(p0.buf, p0.m), lists(buf, mode == TG_PUBLISH ? 0 : used), r, mode,
                   ctx->mapped_dev(seq), seq);
        if (mode != TG_ROUND) q.push_back(seq);
        if (mode == TG_PUBLISH) return;
        at.push_back({buf, used++, held});
        launched++;
    };
    u64 rows_next = 0;
    *total = 0;
    while (true) {
        while (launched < it + 2 + TG_DEPTH && (max_it <= 0 || launched < max_it)) {
            // the buffer's rounds are full, or its entries will be: then the rounds launched are waited for first
            const bool full = used == TG_META || (used >= 2 && buf == use_buf && use + (launched - it + 1) * growth > a.region);
            if (full && launched > it) break;
            if (full) turn(used, (u32)launched + 1);
            launch(launched == it ? TG_ROUND : TG_BOTH);   // the last round may be known already
        }
        if (q.empty()) launch(TG_PUBLISH);   // nothing follows the last round yet
        const u64 seq = q.front();
        q.pop_front();
        ctx->wait_mapped(seq);
        const volatile u64 *m = ctx->mapped_host(seq);
        const u64 nn = m[0];
        if (m[3]) {   // round it + 1 found its region full: again, in the other buffer
            const Round v = at[2];   // at[0], at[1]: rounds it - 1 and it
            ctx->sync();             // the rounds queued behind it have passed without work
            q.clear();
            at.resize(2);
            launched = it;
            if (v.m < 2) return -1;
            buf = v.buf;
            held = v.held;
            turn(v.m, (u32)(it + 1));
            continue;
        }
        it++;
        *total += nn;
        if (at[1].buf == use_buf && m[4] > use) growth = (m[4] - use) * 5 / 4;
        use = m[4];
        use_buf = at[1].buf;
        ctx->prof_add_bytes(DLG_K_BITMAP_INSERT, 8.0 * (double)m[2]);
        if (it > 0) *raw += rows_next;   // the join rows of the round before's ends
        rows_next = m[1];
        if (it > 0) at.pop_front();      // round it - 2's lists
        if (it > 0 && (nn == 0 || (max_it > 0 && it >= max_it))) break;
    }
    merge(at[1].buf == buf ? at[1].m + 1 : 0);   // a buffer turned to since has later rounds only
    return it;
}

int tc_rings_run(dlg_ctx *ctx, const TcRows &tr, RowMap &F, int max_it, u64 *total, u64 *raw) {
    // small buffers first: half of F each, which few rounds of few ends never fill
    const u64 most = tg_region_max(F.W, F.blocks[0].wpr);
    u64 r = 0;
    int it = tg_run(ctx, tr, F, max_it, most / 8, total, &r);
    if (it < 0) {   // rings of most of the words, thus few of them: from the start, with room for any
        fill_u32(ctx, F.words.p, F.nwords, 0u);
        r = 0;
        it = tg_run(ctx, tr, F, max_it, most, total, &r);
        if (it < 0) fail(DLG_DEVICE_ERROR, "tc_rings_run: a list buffer does not hold two rounds");
    }
    *raw += r;
    return it;
}

}  // namespace dlg
