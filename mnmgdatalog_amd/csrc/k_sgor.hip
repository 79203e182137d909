// k_sgor.hip -- SG's rounds as two row ORs.
//
// SG is symmetric (both rules are, sg.cu:300-375), so its maps are: with Δ(a, b)
// as row a of D, a round is
//     X row x = OR over the predecessors a of x of D row a      (the first join)
//     T = X transposed                                          (row b: the x of T(b, x))
//     N row y = (OR over the predecessors b of y of T row b) & ~(F row y)
//
//   sg_or_x_k   a workgroup makes 512 rows x by one chunk of 32 words of X in LDS
//               and writes it transposed: 16 words (a segment) of each of T's
//               1,024 rows b.  It reads a source row's chunk once, by 8 lanes,
//               and ORs it into the rows x of its edges (LDS atomics on the
//               words that hold something); the edges stand by tile and source
//               row (`list`).
//   sg_or_n_k   a wave makes a row y by a group of 8 chunks: a kilobyte of each
//               predecessor's T row and of F's, all in flight, then F and D
// D carries a flag per row and chunk and T one per row and segment: what is not
// flagged is neither read nor valid, so nothing is cleared between rounds, and
// the rounds are queued ahead of the host (round r publishes r - 1's totals).
//
// Bound by the maps' traffic (the second OR: 610 MB a round, 192 us, of which
// 143 at the rate of a copy) and by the LDS steps per edge and chunk (the first:
// 290 MB, 173 us).  What the first one took before, on the same rounds: a
// gather of each row's predecessors 250-300 us, as each chunk is then read from
// L2 once per edge; with the 32 x 32-bit transposition by lane exchanges 300.
// An XCD takes a contiguous eighth of the rows, chunk by chunk: a mesh's
// predecessors are near, so their chunks are in its L2.
//
// Whole calls against the row kernels of k_sgrows.hip, which walk Δ's bits and
// OR each one's successors into a row in LDS: the tetrahedral mesh of 46,656
// vertices (52 rounds, 2.0e9 tuples) 49 -> 26 ms; meshes of 729 and 64,000
// vertices 0.88 -> 0.53 and 89 -> 38; power-law graphs of 40,000 ids 88 -> 5.5 and
// of 131,000 ids 195 -> 26; sparse ranges of 175,000 ids (269 rounds) 504 -> 308;
// a ladder of 3,000 rounds 137 -> 42; none of 30 inputs slower.
#include "dlg_internal.h"

#include <algorithm>
#include <deque>

namespace dlg {

constexpr int SO_L = 8;          // lanes per chunk
constexpr u32 SO_CW = 32;        // words per chunk (8 lanes x 4)
constexpr int SX_T = 512, SX_LOG = 9, SX_R = 1 << SX_LOG, SX_SUB = SX_T / SO_L;   // first OR: threads, rows per tile, sub-groups
static_assert(!sg_or_takes(1ull << (30 - SX_LOG)), "an edge of a tile and two flags in 32 bits");
constexpr u32 SO_SEG = SX_R / 32;       // words of T per row and tile: a segment, with a flag of its own
constexpr u32 SO_G = SO_SEG / 2;        // chunks per group: 16 segments, a wave's uint4s
constexpr int SN_T = 256, SN_W = SN_T / WAVE, SN_RW = 8, SN_R = SN_W * SN_RW;   // second OR: threads, waves, rows per wave and workgroup
constexpr u32 SO_LONG = 64;      // predecessors above which a workgroup of the second OR shares the row
constexpr u32 SO_XCD = 8;
constexpr int SO_SETS = 4, SO_SLOT = 8;
constexpr u32 SO_SLOTS = 64;
constexpr int SO_DEPTH = 3;    // rounds queued ahead of the host
static_assert(SX_R <= SX_T, "a thread transposes a block");
static_assert(SO_G * SO_CW == 4 * WAVE && SO_G == SO_L, "a wave reads a group of a row");
static_assert(SO_DEPTH + 2 <= dlg_ctx::MAPPED_SLOTS, "every queued round has a mapped slot of its own");

// Counter slots of a round: new tuples, the next first join's rows, the second join's rows.
enum { SO_NN = 0, SO_RAW1 = 1, SO_RAW2 = 2 };

struct SoArgs {
    const u64 *off;          // predecessor lists by row
    const u32 *pred;
    const u32 *list;         // edges (a, x) by x's tile, then a, then x: a << SX_LOG | x within the tile
    const u32 *outdeg;
    u32 *F, *D, *T;
    unsigned char *df;       // D's flags: [chunk][row]
    unsigned char *tf;       // T's flags: [group][row][16 segments]
    unsigned long long *cnt; // SO_SETS sets of SO_SLOTS slots
    u32 *done;               // the round that published an empty one (0: none yet): later work does nothing
    u32 W, wpr, nc;
};

__device__ __forceinline__ bool so_any(const uint4 &v) { return (v.x | v.y | v.z | v.w) != 0u; }
__device__ __forceinline__ void so_or(uint4 &a, const uint4 &b) {
    a.x |= b.x;
    a.y |= b.y;
    a.z |= b.z;
    a.w |= b.w;
}

// The workgroup's unit among nr x nc (row blocks x chunks): an XCD (workgroup
// b goes to XCD b % 8) takes a contiguous eighth of the row blocks, chunk by
// chunk.  False past the end.
__device__ __forceinline__ bool so_unit(u32 b, u32 nr, u32 nc, u32 &row, u32 &ch) {
    const u32 x = b % SO_XCD, i = b / SO_XCD;
    const u32 r0 = (u32)((u64)nr * x / SO_XCD), r1 = (u32)((u64)nr * (x + 1) / SO_XCD), m = r1 - r0;
    if (m == 0 || i >= m * nc) return false;
    ch = i / m;
    row = r0 + i - ch * m;
    return true;
}
static unsigned so_grid(u64 nr, u64 nc) { return (unsigned)(SO_XCD * ((nr + SO_XCD - 1) / SO_XCD) * nc); }

// The sub-group's lanes with a true predicate.
__device__ __forceinline__ u32 so_sub_ballot(bool p) {
    return (u32)(__ballot(p) >> ((threadIdx.x & (WAVE - 1)) & ~(SO_L - 1))) & 0xffu;
}

__device__ __forceinline__ uint4 so_at(const u32 *map, u32 byte) { return *(const uint4 *)((const char *)map + byte); }

template <int NT>
__device__ __forceinline__ void so_add(const SoArgs &a, u32 round, int q, u64 v, u64 *s_red) {   // block-uniform call
#pragma unroll
    for (int d = WAVE / 2; d > 0; d >>= 1) v += __shfl_xor(v, d, WAVE);
    if ((threadIdx.x & (WAVE - 1)) == 0) s_red[threadIdx.x / WAVE] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        u64 t = 0;
        for (int w = 0; w < NT / WAVE; w++) t += s_red[w];
        if (t) atomicAdd(a.cnt + ((u64)(round % SO_SETS) * SO_SLOTS + blockIdx.x % SO_SLOTS) * SO_SLOT + q, (unsigned long long)t);
    }
    __syncthreads();
}

// Publishes round `round` - 1 (round 0: the base rule) and clears the next set.
__device__ __forceinline__ void so_publish(const SoArgs &a, u32 round, u64 *host, u64 seq) {
    if (threadIdx.x >= WAVE) return;
    static_assert(SO_SLOTS == WAVE, "a slice per lane");
    unsigned long long *prev = a.cnt + ((u64)((round - 1) % SO_SETS) * SO_SLOTS + threadIdx.x) * SO_SLOT;
    unsigned long long *next = a.cnt + ((u64)((round + 1) % SO_SETS) * SO_SLOTS + threadIdx.x) * SO_SLOT;
    u64 t[3];
#pragma unroll
    for (int q = 0; q < 3; q++) {
        t[q] = prev[q];
        next[q] = 0;
#pragma unroll
        for (int d = WAVE / 2; d > 0; d >>= 1) t[q] += __shfl_xor(t[q], d, WAVE);
    }
    if (threadIdx.x == 0) {
        if (round > 1 && t[SO_NN] == 0 && *a.done == 0u) *a.done = round;
        for (int q = 0; q < 3; q++) host[q] = t[q];
        __threadfence_system();
        *(volatile u64 *)(host + dlg_ctx::MAPPED_SEQ) = seq;
        __threadfence_system();
    }
}

// One step of a 32 x 32-bit transposition: swaps bit J of the row and of the column.
template <int J>
__device__ __forceinline__ void so_swap(u32 (&w)[32]) {
    constexpr u32 m = J == 16 ? 0x0000ffffu : J == 8 ? 0x00ff00ffu : J == 4 ? 0x0f0f0f0fu : J == 2 ? 0x33333333u : 0x55555555u;
#pragma unroll
    for (int i = 0; i < 32; i++) {
        if (i & J) continue;
        const u32 lo = w[i], hi = w[i + J];
        w[i] = (lo & m) | ((hi << J) & ~m);
        w[i + J] = ((lo >> J) & m) | (hi & ~m);
    }
}

// T from D: SX_R rows x and a chunk.
__global__ __launch_bounds__(SX_T, 4) void sg_or_x_k(SoArgs a, u32 round, int publish_only, u64 *host, u64 seq) {
    // The tile, row by row, the first pairs of the sub-group's lanes side by side, then their second pairs; then
    // T's 1,024 rows, word by word: [word][32 rows][33], the words TS apart, which spreads both the transposed
    // blocks' rows and the segments' words over the 64 banks.
    constexpr int RS = (int)SO_CW + 2, TS = 33 * (int)SO_CW + 4;
    constexpr int LDSW = SX_R * RS > (int)SO_SEG * TS ? SX_R * RS : (int)SO_SEG * TS;
    __shared__ __align__(16) u32 tile[LDSW];
    __shared__ u64 s_red[SX_T / WAVE];
    if (blockIdx.x == 0) {
        so_publish(a, round, host, seq);
        return;
    }
    // this launch's publisher may set `done` meanwhile, which must not part a workgroup's waves: earlier rounds' only
    const u32 stop = *(volatile const u32 *)a.done;
    if (publish_only || (stop && stop < round)) return;
    u32 tr, ch;
    if (!so_unit(blockIdx.x - 1, (a.W + SX_R - 1) / SX_R, a.nc, tr, ch)) return;
    const int l = threadIdx.x % SO_L, sub = threadIdx.x / SO_L, s0 = (threadIdx.x & (WAVE - 1)) & ~(SO_L - 1);
    const u32 x0 = tr * SX_R, cw = ch * SO_CW + 4 * l, wb = a.wpr * 4;
    const u32 cb = min(cw, a.wpr - 4) * 4;   // the lane's words in the row (past it: others, for rows of T past the last)
    const unsigned char *df = a.df + (u64)ch * a.W;
    // the rows b of T that the chunk's columns become, PL lanes a row
    constexpr int PL = SO_SEG / 4, NOUT = 32 * (int)SO_CW / (SX_T / PL);
    const u32 b0 = ch * SO_CW * 32, g = tr / 16, fi = tr % 16;
    const int q4 = 4 * (threadIdx.x % PL), lane = threadIdx.x & (WAVE - 1);
    u32 od[NOUT];
#pragma unroll
    for (int i = 0; i < NOUT; i++) od[i] = a.outdeg[min(b0 + threadIdx.x / PL + i * (SX_T / PL), a.W - 1)];
    // a sub-group takes a contiguous part of the tile's edges, which are in the order of their source rows
    const u64 e0 = a.off[x0], ne = a.off[min(x0 + SX_R, a.W)] - e0, part = (ne + SX_SUB - 1) / SX_SUB;
    const u32 *list = a.list + e0;
    u64 e = min((u64)sub * part, ne);
    const u64 ee = min(e + part, ne);
    // lane l holds the entries l and 8 + l of a turn's 16: source row << 9 | row of the tile.  A turn's are read
    // two turns ahead, their rows' flags one turn ahead.
    auto entry = [&](u64 at) { return list[min(at, ne - 1)]; };
    u32 c0 = 0, c1 = 0, f0 = 0, f1 = 0, n0 = 0, n1 = 0;
    if (ne) {   // block-uniform
        c0 = entry(e + l);
        c1 = entry(e + SO_L + l);
        n0 = entry(e + 2 * SO_L + l);
        n1 = entry(e + 3 * SO_L + l);
        f0 = df[c0 >> SX_LOG];
        f1 = df[c1 >> SX_LOG];
    }
    for (int i = threadIdx.x; i < SX_R * RS; i += SX_T) tile[i] = 0;
    __syncthreads();
    bool some = false;
    uint4 last = make_uint4(0u, 0u, 0u, 0u);   // the chunk of the source row at hand
    u32 before = 0xffffffffu;                  // the entry before the turn's first (lane 0's is used)
    for (; __ballot(e < ee); e += 2 * SO_L) {
        const u32 a0 = (u32)__shfl((int)c0, s0 + (l + SO_L - 1) % SO_L, WAVE), a1 = (u32)__shfl((int)c1, s0 + (l + SO_L - 1) % SO_L, WAVE);
        const bool new0 = ((l ? a0 : before) ^ c0) >> SX_LOG, new1 = ((l ? a1 : a0) ^ c1) >> SX_LOG;
        before = a1;
        if (f0 && e + l < ee) c0 |= new0 ? 0xc0000000u : 0x80000000u;   // to be taken; to be read
        if (f1 && e + SO_L + l < ee) c1 |= new1 ? 0xc0000000u : 0x80000000u;
        u32 en[2 * SO_L];
        uint4 v[2 * SO_L];
#pragma unroll
        for (int k = 0; k < 2 * SO_L; k++) en[k] = (u32)__shfl((int)(k < SO_L ? c0 : c1), s0 + k % SO_L, WAVE);
        __builtin_amdgcn_sched_barrier(0);   // all in flight before the first is used
#pragma unroll
        for (int k = 0; k < 2 * SO_L; k++)
            if (en[k] & 0x40000000u) v[k] = so_at(a.D, __umul24((en[k] & 0x3fffffffu) >> SX_LOG, wb) + cb);
        c0 = n0;
        c1 = n1;
        f0 = df[c0 >> SX_LOG];
        f1 = df[c1 >> SX_LOG];
        n0 = entry(e + 4 * SO_L + l);
        n1 = entry(e + 5 * SO_L + l);
#pragma unroll
        for (int k = 0; k < 2 * SO_L; k++) {
            if (en[k] & 0x40000000u) last = v[k];
            if ((int)en[k] < 0 && so_any(last)) {
                unsigned long long *t = (unsigned long long *)(tile + __umul24(en[k] & (SX_R - 1), RS) + 2 * l);
                atomicOr(t, (unsigned long long)last.y << 32 | last.x);
                atomicOr(t + 8, (unsigned long long)last.w << 32 | last.z);
                some = true;
            }
        }
    }
    const bool any = __syncthreads_or(some);
    u64 raw = 0;
    if (any) {   // a thread transposes the 32 x 32 bits of 32 rows R and word C
        const u32 R = threadIdx.x / SO_CW, C = threadIdx.x % SO_CW, word = C / 16 * 2 + (C % 16 / 2) * 4 + C % 2;
        u32 w[32];
        if (threadIdx.x < SX_R) {
#pragma unroll
            for (int i = 0; i < 32; i++) w[i] = tile[(R * 32 + i) * RS + C];
        }
        __syncthreads();
        if (threadIdx.x < SX_R) {
            so_swap<16>(w);
            so_swap<8>(w);
            so_swap<4>(w);
            so_swap<2>(w);
            so_swap<1>(w);
#pragma unroll
            for (int i = 0; i < 32; i++) tile[R * TS + word * 33 + i] = w[i];
        }
        __syncthreads();
    }
    // T's segments out, four words a lane, flagged when not empty
    const bool fits = tr * SO_SEG + q4 < a.wpr;   // the last tile may reach past the row
#pragma unroll
    for (int i = 0; i < NOUT; i++) {
        const u32 j = threadIdx.x / PL + i * (SX_T / PL), b = b0 + j;
        uint4 w = make_uint4(0u, 0u, 0u, 0u);
        if (any && b < a.W) {
            const u32 *t = &tile[q4 * TS + j / 32 * 33 + j % 32];
            w = make_uint4(t[0], t[TS], t[2 * TS], t[3 * TS]);
        }
        const bool f = ((u32)(__ballot(so_any(w)) >> (lane & ~(PL - 1))) & ((1u << PL) - 1u)) != 0u;
        if (f && fits) *(uint4 *)((char *)a.T + (b * wb + (tr * SO_SEG + q4) * 4)) = w;   // no bits past row W
        raw += (u64)(__popc(w.x) + __popc(w.y) + __popc(w.z) + __popc(w.w)) * od[i];
        if (q4 == 0 && b < a.W) a.tf[((u64)g * a.W + b) * 16 + fi] = (unsigned char)f;
    }
    so_add<SX_T>(a, round, SO_RAW2, raw, s_red);
}

// The 16 flags of a row's group of segments, a bit each.
__device__ __forceinline__ u32 so_flags(const unsigned char *p) {
    const uint4 v = *(const uint4 *)p;
    const u32 w[4] = {v.x, v.y, v.z, v.w};
    u32 r = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) r |= ((w[q] & 1u) | ((w[q] >> 7) & 2u) | ((w[q] >> 14) & 4u) | ((w[q] >> 21) & 8u)) << (4 * q);
    return r;
}

// ORs the group's words of one row's predecessors into acc: lane j holds row
// offset `zoff` (bytes) and flags `f`; `fb` is the flag of this lane's words (an
// unflagged segment holds what an earlier round left), `none` a row of zeros.
__device__ __forceinline__ void so_gather_t(uint4 &acc, u32 zoff, u32 f, u32 fb, const u32 *map, u32 cb, u32 none) {
    u64 m = __ballot(f != 0u);
    while (m) {
        uint4 v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int j = m ? __ffsll((unsigned long long)m) - 1 : 0;
            const u32 ff = m ? (u32)__builtin_amdgcn_readlane((int)f, j) : 0u;
            const u32 zz = (u32)__builtin_amdgcn_readlane((int)zoff, j);
            m &= m - 1;   // 0 stays 0
            v[k] = so_at(map, (ff >> fb) & 1u ? zz + cb : none);
        }
#pragma unroll
        for (int k = 0; k < 4; k++) so_or(acc, v[k]);
    }
}

// N from T: SN_R rows y and a group; a wave takes a row's group at a time, a
// kilobyte of each predecessor's row and of F.
__global__ __launch_bounds__(SN_T) void sg_or_n_k(SoArgs a, u32 round) {
    __shared__ u64 s_red[SN_W];
    __shared__ u32 s_long[SN_R];
    __shared__ u32 s_nlong;
    __shared__ __align__(16) u32 s_acc[4 * WAVE];
    if (*a.done) return;
    u32 rb, g;
    if (!so_unit(blockIdx.x, (a.W + SN_R - 1) / SN_R, (a.nc + SO_G - 1) / SO_G, rb, g)) return;
    const int lane = threadIdx.x & (WAVE - 1), wv = threadIdx.x / WAVE, k8 = lane % 8, r8 = lane / 8;
    const u32 y0 = rb * SN_R + (u32)wv * SN_RW, yl = y0 + (u32)r8;
    const unsigned char *tf = a.tf + (u64)g * a.W * 16;
    const u32 wb = a.wpr * 4, none = a.W * wb;   // a row of zeros behind the map
    const u32 cw = g * SO_G * SO_CW + 4 * (u32)lane, cb = min(cw, a.wpr - 4) * 4, fb = 4 * (u32)lane / SO_SEG;
    const bool in_row = cw < a.wpr;
    if (threadIdx.x == 0) s_nlong = 0;
    __syncthreads();
    // lane 8 r + k: predecessor k of row r, its flags
    u64 p0 = 0;
    u32 len = 0, zo = 0, f = 0, outd = 0;
    bool lng = false;
    if (yl < a.W) {
        p0 = a.off[yl];
        const u64 d = a.off[yl + 1] - p0;
        outd = a.outdeg[yl];
        len = (u32)min(d, (u64)SO_LONG + 1);
        if (len > SO_LONG) {
            if (k8 == 0) s_long[atomicAdd(&s_nlong, 1u)] = yl - rb * SN_R;
            lng = true;
            len = 0;
        }
        if (k8 < (int)len) {
            const u32 z = a.pred[p0 + k8];
            zo = z * wb;
            f = so_flags(tf + (u64)z * 16);
        }
    }
    u64 nn = 0, raw = 0;
    bool flag = false;   // lane 8 r + c: chunk c of row r holds new tuples
    // the new words of row y of `acc`, into F and D
    auto update = [&](const uint4 &acc, const uint4 &o, u32 y, u32 od) {
        const u64 at = (u64)y * a.wpr + cw;
        const uint4 n = make_uint4(acc.x & ~o.x, acc.y & ~o.y, acc.z & ~o.z, acc.w & ~o.w);
        const u64 b = __ballot(so_any(n));
        if (so_any(n)) *(uint4 *)(a.F + at) = make_uint4(o.x | n.x, o.y | n.y, o.z | n.z, o.w | n.w);
        if (((b >> (lane & ~7)) & 0xffull) && in_row) *(uint4 *)(a.D + at) = n;   // a flagged chunk is written whole
        const u32 c = (u32)(__popc(n.x) + __popc(n.y) + __popc(n.z) + __popc(n.w));
        nn += c;
        raw += (u64)c * od;
        return b;
    };
#pragma unroll 2
    for (int r = 0; r < SN_RW; r++) {
        const u32 fr = f, any = (u32)(__ballot(fr != 0u) >> (8 * r)) & 0xffu, n = (u32)__builtin_amdgcn_readlane((int)len, 8 * r);
        if (any == 0 && n <= 8) continue;   // wave-uniform
        const u32 y = y0 + (u32)r;
        uint4 acc = make_uint4(0u, 0u, 0u, 0u), o = acc, v[8];
        if (in_row) o = *(const uint4 *)(a.F + (u64)y * a.wpr + cw);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const u32 fk = (u32)__builtin_amdgcn_readlane((int)f, 8 * r + k), zk = (u32)__builtin_amdgcn_readlane((int)zo, 8 * r + k);
            v[k] = so_at(a.T, (fk >> fb) & 1u ? zk + cb : none);
        }
#pragma unroll
        for (int k = 0; k < 8; k++) so_or(acc, v[k]);
        if (n > 8) {   // the others
            const u64 p = __shfl(p0, 8 * r, WAVE);
            const bool in = 8 + lane < (int)n;
            const u32 z = in ? a.pred[p + 8 + lane] : 0u;
            so_gather_t(acc, z * wb, in ? so_flags(tf + (u64)z * 16) : 0u, fb, a.T, cb, none);
        }
        if (!in_row) acc = make_uint4(0u, 0u, 0u, 0u);
        const u64 b = update(acc, o, y, (u32)__builtin_amdgcn_readlane((int)outd, 8 * r));
        if (r8 == r) flag = ((b >> (8 * k8)) & 0xffull) != 0ull;
    }
    if (yl < a.W && !lng && g * SO_G + (u32)k8 < a.nc) a.df[(u64)(g * SO_G + (u32)k8) * a.W + yl] = flag;
    __syncthreads();
    const u32 nl = s_nlong;
    for (u32 i = 0; i < nl; i++) {   // block-uniform: every wave takes a part of a long row
        const u32 y = rb * SN_R + s_long[i];
        const u64 q0 = a.off[y], q1 = a.off[y + 1];
        if (wv == 0) *(uint4 *)&s_acc[4 * lane] = make_uint4(0u, 0u, 0u, 0u);
        __syncthreads();
        uint4 acc = make_uint4(0u, 0u, 0u, 0u);
        for (u64 q = q0 + (u64)wv * WAVE; q < q1; q += SN_T) {   // wave-uniform
            const bool in = q + lane < q1;
            const u32 z = in ? a.pred[q + lane] : 0u;
            so_gather_t(acc, z * wb, in ? so_flags(tf + (u64)z * 16) : 0u, fb, a.T, cb, none);
        }
        if (so_any(acc) && in_row) {
            atomicOr(&s_acc[4 * lane], acc.x);
            atomicOr(&s_acc[4 * lane + 1], acc.y);
            atomicOr(&s_acc[4 * lane + 2], acc.z);
            atomicOr(&s_acc[4 * lane + 3], acc.w);
        }
        __syncthreads();
        if (wv == 0) {
            uint4 o = make_uint4(0u, 0u, 0u, 0u);
            if (in_row) o = *(const uint4 *)(a.F + (u64)y * a.wpr + cw);
            const u64 b = update(*(const uint4 *)&s_acc[4 * lane], o, y, a.outdeg[y]);
            if (lane < (int)SO_G && g * SO_G + (u32)lane < a.nc)
                a.df[(u64)(g * SO_G + (u32)lane) * a.W + y] = ((b >> (8 * lane)) & 0xffull) != 0ull;
        }
        __syncthreads();   // s_acc is rewritten for the next one
    }
    so_add<SN_T>(a, round, SO_NN, nn, s_red);
    so_add<SN_T>(a, round, SO_RAW1, raw, s_red);
}

// D's flags, tuples and next first join's rows after the base rule (round 0).
__global__ __launch_bounds__(SN_T) void so_base_k(SoArgs a) {
    __shared__ u64 s_red[SN_T / WAVE];
    u64 nn = 0, raw = 0;
    const u64 tasks = (u64)a.W * a.nc, stride = (u64)gridDim.x * (SN_T / SO_L);
    const int l = threadIdx.x % SO_L, s0 = (threadIdx.x & (WAVE - 1)) & ~(SO_L - 1);
    for (u64 t0 = (u64)blockIdx.x * (SN_T / SO_L); t0 < tasks; t0 += stride) {   // block-uniform
        const u64 t = t0 + threadIdx.x / SO_L;
        const u32 y = t < tasks ? (u32)(t / a.nc) : 0u, ch = t < tasks ? (u32)(t - (u64)y * a.nc) : 0u;
        const u32 cw = ch * SO_CW + 4 * l;
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        if (t < tasks && cw < a.wpr) v = *(const uint4 *)(a.D + (u64)y * a.wpr + cw);
        const bool has = ((u32)(__ballot(so_any(v)) >> s0) & 0xffu) != 0u;
        if (l == 0 && t < tasks) a.df[(u64)ch * a.W + y] = has;
        const u32 c = (u32)(__popc(v.x) + __popc(v.y) + __popc(v.z) + __popc(v.w));
        nn += c;
        if (c) raw += (u64)c * a.outdeg[y];
    }
    so_add<SN_T>(a, 0, SO_NN, nn, s_red);
    so_add<SN_T>(a, 0, SO_RAW1, raw, s_red);
}

__global__ void so_hist_k(const u64 *rows, u64 n, u32 lo, u32 *indeg, u32 *outdeg) {
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        atomicAdd(outdeg + (tkey(rows[i]) - lo), 1u);
        atomicAdd(indeg + (tval(rows[i]) - lo), 1u);
    }
}
__global__ void so_fill_k(const u64 *rows, u64 n, u32 lo, const u64 *off, u32 *indeg, u32 *pred) {
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const u32 y = tval(rows[i]) - lo;
        pred[off[y] + atomicSub(indeg + y, 1u) - 1u] = tkey(rows[i]) - lo;
    }
}

// Tuples (tile of x, a << SX_LOG | x within the tile) of the edges (a, x), and the sorted ones' second halves.
__global__ void so_key_k(const u64 *rows, u64 n, u32 lo, u64 *out) {
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const u32 x = tval(rows[i]) - lo;
        out[i] = (u64)(x >> SX_LOG) << 32 | ((tkey(rows[i]) - lo) << SX_LOG | (x & (SX_R - 1)));
    }
}
__global__ void so_list_k(const u64 *in, u64 n, u32 *list) {
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) list[i] = (u32)in[i];
}

// Words of `zero`: the counters, T's flags, the degrees (in: W, out: W) and `done`.
constexpr u64 SO_COUNT_WORDS = (u64)SO_SETS * SO_SLOTS * SO_SLOT;
static u64 so_chunks(const Bitmap &F) { return (F.wpr + SO_CW - 1) / SO_CW; }
static u64 so_flag_words(const Bitmap &F) { return F.W * ((so_chunks(F) + SO_G - 1) / SO_G) * 2; }

void sg_or_setup(dlg_ctx *ctx, const u64 *edges, u64 n, const Bitmap &F, SgOr &so) {
    if (F.wpr % 4 || !sg_or_takes(F.W)) fail(DLG_INVALID_INPUT, "sg_or_setup: a map of rows of whole uint4s");
    const u64 W = F.W, tfw = so_flag_words(F), zw = SO_COUNT_WORDS + tfw + (2 * W + 2) / 2;
    DBuf<u64> key(ctx, n ? n : 1), tmp(ctx);
    so.zero.ensure(zw);
    so.off.ensure(W + 1);
    so.df.ensure(W * so_chunks(F));
    so.pred.ensure(n ? n : 1);
    so.list.ensure(n ? n : 1);
    so.T.ensure(F.nwords + 4);   // and four words of zeros, read for what is not flagged
    fill_u32(ctx, so.T.p + F.nwords, 4, 0u);
    fill_u64(ctx, so.zero.p, zw, 0ull);
    u32 *indeg = (u32 *)(so.zero.p + SO_COUNT_WORDS + tfw), *outdeg = indeg + W;
    DLG_LAUNCH(ctx, DLG_K_MISC, 16.0 * n, so_hist_k, sgrid(ctx, n), ctx->block_size, 0, edges, n, F.lo, indeg, outdeg);
    scan_u32_u64_async(ctx, indeg, W, so.off.p, so.off.p + W);
    DLG_LAUNCH(ctx, DLG_K_MISC, 20.0 * n, so_fill_k, sgrid(ctx, n), ctx->block_size, 0, edges, n, F.lo,
               (const u64 *)so.off.p, indeg, so.pred.p);
    DLG_LAUNCH(ctx, DLG_K_MISC, 16.0 * n, so_key_k, sgrid(ctx, n), ctx->block_size, 0, edges, n, F.lo, key.p);
    const u32 bounds[4] = {0, ((u32)W - 1) >> SX_LOG, 0, ((u32)W << SX_LOG) - 1};
    radix_sort(ctx, key, n, tmp, 0, bounds);
    DLG_LAUNCH(ctx, DLG_K_MISC, 12.0 * n, so_list_k, sgrid(ctx, n), ctx->block_size, 0, (const u64 *)key.p, n, so.list.p);
}

int sg_or_run(dlg_ctx *ctx, SgOr &so, Bitmap &F, Bitmap &D, int max_it, u64 *total, u64 *raw) {
    if (D.wpr != F.wpr || D.W != F.W || D.lo != F.lo) fail(DLG_INVALID_INPUT, "sg_or_run: two maps of one geometry");
    SoArgs a;
    a.W = (u32)F.W;
    a.wpr = (u32)F.wpr;
    a.nc = (u32)so_chunks(F);
    const u32 ng = (a.nc + SO_G - 1) / SO_G;
    a.cnt = (unsigned long long *)so.zero.p;
    a.tf = (unsigned char *)(so.zero.p + SO_COUNT_WORDS);
    a.outdeg = (const u32 *)(so.zero.p + SO_COUNT_WORDS + so_flag_words(F)) + a.W;
    a.done = (u32 *)a.outdeg + a.W;
    a.F = F.words.p;
    a.D = D.words.p;
    a.T = so.T.p;
    a.df = so.df.p;
    a.off = so.off.p;
    a.pred = so.pred.p;
    a.list = so.list.p;
    DLG_LAUNCH(ctx, DLG_K_MISC, 4.0 * F.nwords, so_base_k,
               (unsigned)std::min<u64>(((u64)a.W * a.nc * SO_L + SN_T - 1) / SN_T, (u64)ctx->num_cus * 8), SN_T, 0, a);
    const unsigned gx = 1 + so_grid((a.W + SX_R - 1) / SX_R, a.nc), gn = so_grid((a.W + SN_R - 1) / SN_R, ng);
    std::deque<u64> q;   // sequence numbers of the rounds not read yet, from round `it` + 1 on
    int launched = 0, it = -1;
    auto launch = [&](bool publish_only) {
        const u32 r = (u32)launched + 1;
        const u64 seq = ++ctx->mapped_seq;
        DLG_LAUNCH(ctx, DLG_K_BITMAP_INSERT, publish_only ? 0.0 : 8.0 * F.nwords, sg_or_x_k, publish_only ? 1u : gx, SX_T, 0, a, r,
                   publish_only ? 1 : 0, ctx->mapped_dev(seq), seq);
        q.push_back(seq);
        if (publish_only) return;
        DLG_LAUNCH(ctx, DLG_K_BITMAP_INSERT, 16.0 * F.nwords, sg_or_n_k, gn, SN_T, 0, a, r);
        launched++;
    };
    u64 rows_next = 0;
    *total = 0;
    while (true) {
        while (launched < it + 2 + SO_DEPTH && (max_it <= 0 || launched < max_it)) launch(false);
        if (q.empty()) launch(true);   // the last round asked for
        const u64 seq = q.front();
        q.pop_front();
        ctx->wait_mapped(seq);
        const volatile u64 *m = ctx->mapped_host(seq);
        const u64 nn = m[SO_NN];
        it++;
        *total += nn;
        if (it > 0) *raw += rows_next + m[SO_RAW2];   // both joins of this round
        rows_next = m[SO_RAW1];
        if (it > 0 && (nn == 0 || (max_it > 0 && it >= max_it))) break;
    }
    return it;
}

}  // namespace dlg
