// k_prims.hip -- data-parallel primitives for the fixpoint engine on gfx950.
//
// Replaces the Thrust calls of the reference (sort/unique/set_difference/
// merge/reduce/exclusive_scan; sites in tc.cu:177-283, sg.cu:150-368,
// wcc.cu:163-463, single_join.cu:165-264, common/join.cu:72-74) with
// hand-written kernels:
//   * exclusive scan       reduce -> scan of block sums -> apply
//   * radix sort           LSD, reduce-then-scan per digit, wave-match ranking
//                          (64-lane ballots), LDS staging for coalesced scatter;
//                          digits run over a compacted key (hi - min_hi, lo - min_lo)
//                          so only the bits that vary are sorted
//   * select (compaction)  unique / unique minus diagonal / unique minus a sorted
//                          set / set difference / key-run heads; flags are
//                          ballot words, offsets are a block-sum scan
//   * merge                rank-by-binary-search scatter (a first on ties)
#include "dlg_internal.h"

#include <algorithm>
#include <unistd.h>

namespace dlg {

// =============================================================== fills / copies
__global__ void fill_u64_k(u64 *p, u64 n, u64 v) {
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    u64 stride = (u64)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}
__global__ void fill_u32_k(u32 *p, u64 n, u32 v) {
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    u64 stride = (u64)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}
__global__ void copy_u64_k(u64 *dst, const u64 *src, u64 n) {
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    u64 stride = (u64)gridDim.x * blockDim.x;
    for (; i < n; i += stride) dst[i] = src[i];
}

void fill_u64(dlg_ctx *ctx, u64 *p, u64 n, u64 v) {
    if (!n) return;
    DLG_LAUNCH(ctx, DLG_K_MISC, 8.0 * n, fill_u64_k, sgrid(ctx, n), ctx->block_size, 0, p, n, v);
}
void fill_u32(dlg_ctx *ctx, u32 *p, u64 n, u32 v) {
    if (!n) return;
    DLG_LAUNCH(ctx, DLG_K_MISC, 4.0 * n, fill_u32_k, sgrid(ctx, n), ctx->block_size, 0, p, n, v);
}
void copy_u64(dlg_ctx *ctx, u64 *dst, const u64 *src, u64 n) {
    if (!n) return;
    DLG_LAUNCH(ctx, DLG_K_MISC, 16.0 * n, copy_u64_k, sgrid(ctx, n), ctx->block_size, 0, dst, src, n);
}

// =============================================================== pack / unpack
// Tuple t = ((col_a ^ 0x80000000) << 32) | (col_b ^ 0x80000000): u64 order is
// the signed lexicographic order of the reference's set_cmp.
__global__ void pack_k(const int2 *rows, u64 n, int orient, u64 *out) {
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    u64 stride = (u64)gridDim.x * blockDim.x;
    for (; i < n; i += stride) {
        int2 r = rows[i];
        u32 a = (u32)r.x ^ 0x80000000u, b = (u32)r.y ^ 0x80000000u;
        out[i] = orient ? tmake(b, a) : tmake(a, b);
    }
}
// Each (a, b) row packed as (a, b) into out and as (b, a) into out_rev and,
// in the same read, the bounds of both columns (as flipped ids) and the
// count of adjacent rows out of signed lexicographic order; one set of
// atomics per workgroup.  (With `miss`, only if it is set.)
__global__ __launch_bounds__(256) void pack_sym_scan_k(const int2 *rows, u64 n, u64 *out, u64 *out_rev, u32 *mm,
                                                       unsigned long long *desc, const u32 *miss) {
    if (miss && *miss == 0u) return;   // the relation may be its own reverse: pack_both_scan_k's (block-uniform)
    u32 mna = 0xffffffffu, mxa = 0u, mnb = 0xffffffffu, mxb = 0u;
    u64 dc = 0;
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const int2 r = rows[i];
        const u32 a = (u32)r.x ^ 0x80000000u, b = (u32)r.y ^ 0x80000000u;
        out[i] = tmake(a, b);
        out_rev[i] = tmake(b, a);
        mna = min(mna, a); mxa = max(mxa, a); mnb = min(mnb, b); mxb = max(mxb, b);
        if (i + 1 < n) {
            const int2 q = rows[i + 1];
            dc += r.x > q.x || (r.x == q.x && r.y > q.y);
        }
    }
#pragma unroll
    for (int d = WAVE / 2; d > 0; d >>= 1) {
        mna = min(mna, (u32)__shfl_xor((int)mna, d, WAVE));
        mxa = max(mxa, (u32)__shfl_xor((int)mxa, d, WAVE));
        mnb = min(mnb, (u32)__shfl_xor((int)mnb, d, WAVE));
        mxb = max(mxb, (u32)__shfl_xor((int)mxb, d, WAVE));
        dc += __shfl_xor(dc, d, WAVE);
    }
    __shared__ u32 sm[4][256 / WAVE];
    __shared__ u64 sd[256 / WAVE];
    const int wave = threadIdx.x / WAVE;
    if ((threadIdx.x & (WAVE - 1)) == 0) {
        sm[0][wave] = mna; sm[1][wave] = mxa; sm[2][wave] = mnb; sm[3][wave] = mxb;
        sd[wave] = dc;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)(blockDim.x / WAVE); w++) {
            mna = min(mna, sm[0][w]); mxa = max(mxa, sm[1][w]);
            mnb = min(mnb, sm[2][w]); mxb = max(mxb, sm[3][w]);
            dc += sd[w];
        }
        // an atomic only where it can still move the bound: after the first
        // workgroups most skip it (a stale read only costs an atomic)
        if (mna < __hip_atomic_load(&mm[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(&mm[0], mna);
        if (mxa > __hip_atomic_load(&mm[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(&mm[1], mxa);
        if (mnb < __hip_atomic_load(&mm[2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(&mm[2], mnb);
        if (mxb > __hip_atomic_load(&mm[3], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(&mm[3], mxb);
        if (dc) atomicAdd(desc, (unsigned long long)dc);
    }
}

// ------------------------------------------- relations that are their own reverse
// A WCC input often lists both directions of every edge, sorted.  It is then its own
// E u E⁻¹, and the reversed copy, its sort and the merge are for nothing (R-MAT-23,
// 2.6e8 rows: 13.2 -> 4.8 ms for the whole call).  Whether it is, in one read: the rows are in strictly
// ascending order, and {(a, b) : a < b} and {(b, a) : a > b} are the same set, which
// two products over the rows tell,
//     prod (r - min(a, b) - s max(a, b))  mod p = 2^61 - 1,  once over a < b, once over a > b.
// As polynomials in r and s they are the same exactly if the sets are; if not, they
// agree at a point (r, s) drawn after the input is fixed with a probability of at most n / p (Schwartz, Zippel).
// At two points of their own, drawn for every call: 2^-66 for 2^28 rows.
constexpr u64 FP_P = (1ull << 61) - 1;
constexpr int FP_POINTS = 2;
// Rows from which on the look is worth its launches: 80,000 rows in both directions
// 410 -> 250 us, 8,000,000 1.59 -> 1.18 ms; as many in one direction 0.41 and 2.95 ms
// with it and without (within what runs differ by).
constexpr u64 FP_MIN = 1ull << 16;
struct FpPoint {
    u64 r[FP_POINTS], s[FP_POINTS];   // in [0, p)
};
// a b mod p, for a b < 2^124 (its two halves' sum fits in 64 bits); below 2^61 + 8, not always
// below p.  The terms multiplied up are below 2^62 + 2^61, the products they meet below 2^61 + 8.
__device__ __forceinline__ u64 fp_mul(u64 a, u64 b) {
    const u64 lo = a * b, hi = __umul64hi(a, b);
    const u64 t = (lo & FP_P) + ((lo >> 61) | (hi << 3));
    return (t & FP_P) + (t >> 61);
}
__device__ __forceinline__ u64 row_key(int2 r) { return tmake((u32)r.x ^ 0x80000000u, (u32)r.y ^ 0x80000000u); }

// A look before: FP_SAMPLES rows, a wave each, searched for their reverses 64 ways
// at a time (5 reads deep for 2^28 rows); *miss is set if one is not there.  Unsorted
// rows only mislead it, the search stays within [0, n).
constexpr unsigned FP_SAMPLES = 1024, FP_WAVES = 4;
__global__ __launch_bounds__(FP_WAVES * WAVE) void reverse_probe_k(const int2 *rows, u64 n, u32 *miss) {
    const u64 w = (u64)blockIdx.x * FP_WAVES + threadIdx.x / WAVE;
    const u32 lane = threadIdx.x & (WAVE - 1);
    const u64 part = n / FP_SAMPLES, i = w * part + (w * 2654435761ull) % part;   // n >= FP_SAMPLES
    const int2 x = rows[i];
    const u64 want = row_key(make_int2(x.y, x.x));
    u64 lo = 0, hi = n;
    while (lo < hi) {   // the first row >= want is in [lo, hi]; wave-uniform
        const u64 step = (hi - lo + WAVE - 1) / WAVE, at = lo + lane * step;
        const u64 c = (u64)__popcll(__ballot(at < hi && row_key(rows[at < hi ? at : lo]) < want));
        hi = c ? min(hi, lo + c * step) : lo;
        lo = c ? lo + (c - 1) * step + 1 : lo;
    }
    if (lane == 0 && (lo == n || row_key(rows[lo]) != want)) *miss = 1u;
}

// Rows packed as (a, b), with a bit per row that begins a key's run, the count of rows
// not above the one before, and the workgroup's products, unless the look before missed.
// Bound by the products beside the copy (FP_I rows in flight a thread): 2.6e8 rows 1.0
// ms, 4.2 TB/s; the scan that writes both directions takes 1.43.
constexpr int FP_T = 256, FP_I = 4;
__global__ __launch_bounds__(FP_T) void pack_both_scan_k(const int2 *rows, u64 n, u64 *out, u64 *heads, FpPoint at,
                                                        const u32 *miss, u64 *part, unsigned long long *breaks) {
    if (*miss) return;   // set by an earlier launch: the same for all
    u64 up[FP_POINTS], down[FP_POINTS];
#pragma unroll
    for (int k = 0; k < FP_POINTS; k++) up[k] = down[k] = 1;
    u32 dc = 0;
    const u64 tiles = (n + FP_T * FP_I - 1) / (FP_T * FP_I);
    for (u64 tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const u64 base = tile * (FP_T * FP_I) + threadIdx.x;
        int2 v[FP_I], q[FP_I];
#pragma unroll
        for (int j = 0; j < FP_I; j++) {
            const u64 i = base + (u64)j * FP_T;
            v[j] = rows[i < n ? i : n - 1];
            q[j] = rows[i < n && i > 0 ? i - 1 : 0];
        }
#pragma unroll
        for (int j = 0; j < FP_I; j++) {
            const u64 i = base + (u64)j * FP_T;
            const u32 a = (u32)v[j].x ^ 0x80000000u, b = (u32)v[j].y ^ 0x80000000u;
            const u64 x = min(a, b), y = max(a, b);
            if (i < n) out[i] = tmake(a, b);
            dc += i < n && i > 0 && row_key(q[j]) >= tmake(a, b);
            const u64 hm = __ballot(i < n && (i == 0 || q[j].x != v[j].x));   // i: a multiple of 64 in lane 0
            if (threadIdx.x % WAVE == 0 && i < n) heads[i / WAVE] = hm;
            const bool asc = a < b, use = i < n && a != b;
#pragma unroll
            for (int k = 0; k < FP_POINTS; k++) {
                const u64 t = use ? at.r[k] + 2 * FP_P - x - fp_mul(at.s[k], y) : 1ull;
                const u64 m = fp_mul(asc ? up[k] : down[k], t);
                up[k] = asc ? m : up[k];
                down[k] = asc ? down[k] : m;
            }
        }
    }
    __shared__ u64 s_p[2 * FP_POINTS][FP_T / WAVE];
#pragma unroll
    for (int d = WAVE / 2; d > 0; d >>= 1) {
        dc += (u32)__shfl_xor((int)dc, d, WAVE);
#pragma unroll
        for (int k = 0; k < FP_POINTS; k++) {
            up[k] = fp_mul(up[k], __shfl_xor(up[k], d, WAVE));
            down[k] = fp_mul(down[k], __shfl_xor(down[k], d, WAVE));
        }
    }
    if ((threadIdx.x & (WAVE - 1)) == 0) {
#pragma unroll
        for (int k = 0; k < FP_POINTS; k++) {
            s_p[2 * k][threadIdx.x / WAVE] = up[k];
            s_p[2 * k + 1][threadIdx.x / WAVE] = down[k];
        }
        if (dc) atomicAdd(breaks, (unsigned long long)dc);
    }
    __syncthreads();
    if (threadIdx.x < 2 * FP_POINTS) {
        u64 m = 1;
        for (int w = 0; w < FP_T / WAVE; w++) m = fp_mul(m, s_p[threadIdx.x][w]);
        part[(u64)blockIdx.x * 2 * FP_POINTS + threadIdx.x] = m;
    }
}
// The workgroups' products multiplied up, a wave for each; a point at which the two
// differ counts as a break.
__global__ __launch_bounds__(2 * FP_POINTS * WAVE) void fp_fold_k(const u64 *part, u32 nb, const u32 *miss, u64 *breaks) {
    if (*miss) return;
    __shared__ u64 s_m[2 * FP_POINTS];
    const u32 k = threadIdx.x / WAVE, lane = threadIdx.x & (WAVE - 1);
    u64 m = 1;
    for (u32 i = lane; i < nb; i += WAVE) m = fp_mul(m, part[(u64)i * 2 * FP_POINTS + k]);
#pragma unroll
    for (int d = WAVE / 2; d > 0; d >>= 1) m = fp_mul(m, __shfl_xor(m, d, WAVE));
    if (lane == 0) s_m[k] = m % FP_P;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int j = 0; j < FP_POINTS; j++)
            if (s_m[2 * j] != s_m[2 * j + 1]) *breaks += 1;
}

__global__ void unpack_k(const u64 *t, u64 n, int orient, int2 *rows) {
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    u64 stride = (u64)gridDim.x * blockDim.x;
    for (; i < n; i += stride) {
        u64 x = t[i];
        int k = (int)(tkey(x) ^ 0x80000000u), v = (int)(tval(x) ^ 0x80000000u);
        rows[i] = orient ? make_int2(v, k) : make_int2(k, v);
    }
}

void pack_rows(dlg_ctx *ctx, const int32_t *rows, u64 n, int orient, u64 *out) {
    if (!n) return;
    DLG_LAUNCH(ctx, DLG_K_PACK, 16.0 * n, pack_k, sgrid(ctx, n), ctx->block_size, 0,
               (const int2 *)rows, n, orient, out);
}
// Words of a scan: bounds (min a, max a, min b, max b), descents; a miss of the look
// before, the breaks of the scan after it.
constexpr int PS_MISS = 3, PS_BREAKS = 4, PS_WORDS = 5;
__global__ void pack_scan_init_k(u64 *w) {
    u32 *mm = (u32 *)w;
    if (threadIdx.x < 4) mm[threadIdx.x] = threadIdx.x & 1 ? 0u : 0xffffffffu;
    else if (threadIdx.x < 2 + PS_WORDS) w[threadIdx.x - 2] = 0ull;   // words 2 .. PS_WORDS - 1
}
u64 pack_sym_rows_scan(dlg_ctx *ctx, const int32_t *rows, u64 n, u64 *out, u64 *out_rev, u32 *cb, bool *both,
                       DBuf<u64> &heads) {
    cb[0] = cb[1] = cb[2] = cb[3] = 0u;
    *both = false;
    if (!n) return 0;
    DBuf<u64> w(ctx, PS_WORDS);
    const int2 *r = (const int2 *)rows;
    const unsigned g = (unsigned)std::min<u64>((n + 255) / 256, (u64)ctx->num_cus * 8);
    FpPoint at;
    bool look = n >= FP_MIN && getentropy(&at, sizeof(at)) == 0;
    if (look) heads.ensure((n + WAVE - 1) / WAVE);
    while (true) {
        u32 *miss = look ? (u32 *)(w.p + PS_MISS) : nullptr;
        DLG_LAUNCH(ctx, DLG_K_MISC, 0.0, pack_scan_init_k, 1, 64, 0, w.p);
        if (look) {
            for (int k = 0; k < FP_POINTS; k++) {
                at.r[k] %= FP_P;   // 2^64 = 8 mod p: some residues a little likelier, nothing to the bound
                at.s[k] %= FP_P;
            }
            const unsigned gb = (unsigned)std::min<u64>((n + FP_T * FP_I - 1) / (FP_T * FP_I), (u64)ctx->num_cus * 8);
            DBuf<u64> part(ctx, (u64)gb * 2 * FP_POINTS);
            DLG_LAUNCH(ctx, DLG_K_MISC, 0.0, reverse_probe_k, FP_SAMPLES / FP_WAVES, FP_WAVES * WAVE, 0, r, n, miss);
            DLG_LAUNCH(ctx, DLG_K_PACK, 16.0 * n, pack_both_scan_k, gb, FP_T, 0, r, n, out, heads.p, at, (const u32 *)miss, part.p,
                       (unsigned long long *)(w.p + PS_BREAKS));
            DLG_LAUNCH(ctx, DLG_K_MISC, 0.0, fp_fold_k, 1, 2 * FP_POINTS * WAVE, 0, (const u64 *)part.p, (u32)gb,
                       (const u32 *)miss, w.p + PS_BREAKS);
        }
        DLG_LAUNCH(ctx, DLG_K_PACK, 24.0 * n, pack_sym_scan_k, g, 256, 0, r, n, out, out_rev, (u32 *)w.p,
                   (unsigned long long *)(w.p + 2), (const u32 *)miss);
        u64 h[PS_BREAKS + 1];
        ctx->read_scalars(w.p, PS_BREAKS + 1, h);
        if (!look || (u32)h[PS_MISS]) {
            std::memcpy(cb, h, 16);
            return h[2];
        }
        if (h[PS_BREAKS] == 0) {
            *both = true;
            return 0;
        }
        look = false;   // nearly its own reverse, or not in order: the full scan after all
    }
}
void unpack_rows(dlg_ctx *ctx, const u64 *t, u64 n, int orient, int32_t *rows) {
    if (!n) return;
    DLG_LAUNCH(ctx, DLG_K_PACK, 16.0 * n, unpack_k, sgrid(ctx, n), ctx->block_size, 0, t, n, orient,
               (int2 *)rows);
}

// =============================================================== scan
constexpr int SCAN_T = 256, SCAN_I = 8, SCAN_TILE = SCAN_T * SCAN_I;

template <typename T>
__global__ __launch_bounds__(SCAN_T) void scan_reduce_k(const T *in, u64 n, u64 *bsum) {
    __shared__ u64 sc[SCAN_T / WAVE + 1];
    u64 base = (u64)blockIdx.x * SCAN_TILE + (u64)threadIdx.x * SCAN_I;
    u64 s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_I; i++)
        if (base + i < n) s += in[base + i];
    u64 tot;
    block_exclusive_scan<u64>(s, sc, &tot);
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// Block sums scanned in place (exclusive), total to *d_total, by one
// workgroup: each thread sums a contiguous segment of ceil(nb / 1024)
// entries, one block scan of those sums, then each thread rewrites its
// segment from its prefix (the segments stay in cache between the passes).
__global__ __launch_bounds__(1024) void scan_blocks_k(u64 *bsum, u64 nb, u64 *d_total) {
    __shared__ u64 sc[1024 / WAVE + 1];
    const u64 seg = (nb + 1023) / 1024;
    const u64 b0 = (u64)threadIdx.x * seg < nb ? (u64)threadIdx.x * seg : nb;
    const u64 b1 = b0 + seg < nb ? b0 + seg : nb;
    u64 s = 0;
#pragma unroll 8
    for (u64 i = b0; i < b1; i++) s += bsum[i];
    u64 tot;
    u64 run = block_exclusive_scan<u64>(s, sc, &tot);
#pragma unroll 8
    for (u64 i = b0; i < b1; i++) {
        const u64 v = bsum[i];
        bsum[i] = run;
        run += v;
    }
    if (threadIdx.x == 0 && d_total) *d_total = tot;
}

template <typename T>
__global__ __launch_bounds__(SCAN_T) void scan_apply_k(const T *in, u64 n, const u64 *bpre, u64 *out) {
    __shared__ u64 sc[SCAN_T / WAVE + 1];
    u64 base = (u64)blockIdx.x * SCAN_TILE + (u64)threadIdx.x * SCAN_I;
    T v[SCAN_I];
    u64 s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_I; i++) {
        v[i] = base + i < n ? in[base + i] : 0;
        s += v[i];
    }
    u64 ex = block_exclusive_scan<u64>(s, sc, nullptr) + bpre[blockIdx.x];
#pragma unroll
    for (int i = 0; i < SCAN_I; i++) {
        if (base + i < n) out[base + i] = ex;
        ex += v[i];
    }
}

// Block sums scanned in place (exclusive), total to *d_total: one workgroup
// up to SCAN_ONE_WG entries, else reduce -> scan of the partials -> apply.
constexpr u64 SCAN_ONE_WG = 16384;
void scan_blocks(dlg_ctx *ctx, u64 *bsum, u64 nb, u64 *d_total) {
    if (nb <= SCAN_ONE_WG) {
        DLG_LAUNCH(ctx, DLG_K_SCAN, 16.0 * nb, scan_blocks_k, 1, 1024, 0, bsum, nb, d_total);
        return;
    }
    const u64 np = (nb + SCAN_TILE - 1) / SCAN_TILE;
    DBuf<u64> part(ctx, np);
    DLG_LAUNCH(ctx, DLG_K_SCAN, 8.0 * nb + 8.0 * np, scan_reduce_k<u64>, (unsigned)np, SCAN_T, 0,
               (const u64 *)bsum, nb, part.p);
    scan_blocks(ctx, part.p, np, d_total);
    DLG_LAUNCH(ctx, DLG_K_SCAN, 16.0 * nb, scan_apply_k<u64>, (unsigned)np, SCAN_T, 0, (const u64 *)bsum, nb,
               (const u64 *)part.p, bsum);
}

u64 scan_partials(u64 n) {
    u64 nb = (n + SCAN_TILE - 1) / SCAN_TILE;
    return nb ? nb : 1;
}

// A whole scan by one workgroup, for inputs of up to SCAN_SMALL elements:
// one launch of about 3 us instead of three.
constexpr int SCAN_SMALL_T = 1024;
constexpr u64 SCAN_SMALL = (u64)SCAN_SMALL_T * SCAN_I;
template <typename T>
__global__ __launch_bounds__(SCAN_SMALL_T) void scan_small_k(const T *in, u64 n, u64 *out, u64 *d_total) {
    __shared__ u64 sc[SCAN_SMALL_T / WAVE + 1];
    const u64 base = (u64)threadIdx.x * SCAN_I;
    T v[SCAN_I];
    u64 s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_I; i++) {
        v[i] = base + i < n ? in[base + i] : 0;
        s += v[i];
    }
    u64 tot;
    u64 ex = block_exclusive_scan<u64>(s, sc, &tot);   // every read is done before the first write: out may alias in
#pragma unroll
    for (int i = 0; i < SCAN_I; i++) {
        if (base + i < n) out[base + i] = ex;
        ex += v[i];
    }
    if (threadIdx.x == 0 && d_total) *d_total = tot;
}

// The launches of a scan over caller-provided partials (scan_partials(n) u64s).
template <typename T>
static void scan_to_u64_with(dlg_ctx *ctx, const T *in, u64 n, u64 *out, u64 *bsum, u64 *d_total) {
    if (n <= SCAN_SMALL) {
        DLG_LAUNCH(ctx, DLG_K_SCAN, (sizeof(T) + 8.0) * n, scan_small_k<T>, 1, SCAN_SMALL_T, 0, in, n, out, d_total);
        return;
    }
    const u64 nb = scan_partials(n);
    DLG_LAUNCH(ctx, DLG_K_SCAN, (double)sizeof(T) * n + 8.0 * nb, scan_reduce_k<T>, (unsigned)nb, SCAN_T, 0,
               in, n, bsum);
    scan_blocks(ctx, bsum, nb, d_total);
    DLG_LAUNCH(ctx, DLG_K_SCAN, (sizeof(T) + 8.0) * n, scan_apply_k<T>, (unsigned)nb, SCAN_T, 0, in, n,
               (const u64 *)bsum, out);
}

template <typename T>
static void scan_to_u64_async(dlg_ctx *ctx, const T *in, u64 n, u64 *out, u64 *d_total) {
    DBuf<u64> bsum(ctx, scan_partials(n));
    scan_to_u64_with<T>(ctx, in, n, out, bsum.p, d_total);
}

void scan_u32_u64_with(dlg_ctx *ctx, const u32 *in, u64 n, u64 *out, u64 *bsum, u64 *d_total) {
    scan_to_u64_with<u32>(ctx, in, n, out, bsum, d_total);
}

void scan_u32_u64_async(dlg_ctx *ctx, const u32 *in, u64 n, u64 *out, u64 *d_total) {
    scan_to_u64_async<u32>(ctx, in, n, out, d_total);
}

void scan_u64_async(dlg_ctx *ctx, const u64 *in, u64 n, u64 *out, u64 *d_total) {
    scan_to_u64_async<u64>(ctx, in, n, out, d_total);
}

u64 scan_u32_u64(dlg_ctx *ctx, const u32 *in, u64 n, u64 *out) {
    DBuf<u64> tot(ctx, 1);
    scan_u32_u64_async(ctx, in, n, out, tot.p);
    u64 h = 0;
    ctx->read_scalars(tot.p, 1, &h);
    return h;
}

// Exclusive scan of u32 counts into u32 offsets (radix digit counts; sums < 2^32).
__global__ __launch_bounds__(SCAN_T) void scan_reduce32_k(const u32 *in, u64 n, u64 *bsum) {
    __shared__ u64 sc[SCAN_T / WAVE + 1];
    u64 base = (u64)blockIdx.x * SCAN_TILE + (u64)threadIdx.x * SCAN_I;
    u64 s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_I; i++)
        if (base + i < n) s += in[base + i];
    u64 tot;
    block_exclusive_scan<u64>(s, sc, &tot);
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}
__global__ __launch_bounds__(SCAN_T) void scan_apply32_k(u32 *data, u64 n, const u64 *bpre) {
    __shared__ u64 sc[SCAN_T / WAVE + 1];
    u64 base = (u64)blockIdx.x * SCAN_TILE + (u64)threadIdx.x * SCAN_I;
    u32 v[SCAN_I];
    u64 s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_I; i++) {
        v[i] = base + i < n ? data[base + i] : 0;
        s += v[i];
    }
    u64 ex = block_exclusive_scan<u64>(s, sc, nullptr) + bpre[blockIdx.x];
#pragma unroll
    for (int i = 0; i < SCAN_I; i++) {
        if (base + i < n) data[base + i] = (u32)ex;
        ex += v[i];
    }
}
static void scan_u32_inplace(dlg_ctx *ctx, u32 *data, u64 n, DBuf<u64> &bsum) {
    u64 nb = (n + SCAN_TILE - 1) / SCAN_TILE;
    if (nb == 0) nb = 1;
    bsum.ensure(nb);
    DLG_LAUNCH(ctx, DLG_K_SCAN, 4.0 * n, scan_reduce32_k, (unsigned)nb, SCAN_T, 0, data, n,
               bsum.p);
    scan_blocks(ctx, bsum.p, nb, nullptr);
    DLG_LAUNCH(ctx, DLG_K_SCAN, 8.0 * n, scan_apply32_k, (unsigned)nb, SCAN_T, 0, data, n,
               bsum.p);
}

// =============================================================== radix sort
// Tile shapes: 256 threads x 16 keys (4096) for small inputs, 512 threads x
// 32 keys (16384, 128 KiB of LDS staging) for large ones, where longer runs
// per digit make the scatter's writes closer to whole cache lines.
constexpr int RS_SMALL_T = 256, RS_SMALL_I = 16;
constexpr int RS_BIG_T = 512, RS_BIG_I = 32;
constexpr u64 RS_BIG_MIN = 1ull << 21;

struct RadixKey {
    u32 min_hi, min_lo;
    u32 vb;     // bits of (lo - min_lo)
    u32 shift;  // digit position in the compacted key
};

// vb = 0: the value half takes no bits -- every value equal (then lo - min_lo
// is 0 anyway), or a sort by key alone (radix_sort's key_only).
__device__ __forceinline__ u32 radix_digit(u64 x, const RadixKey &k, u32 mask) {
    u64 hi = (u64)(tkey(x) - k.min_hi);
    u64 lo = k.vb ? (u64)(tval(x) - k.min_lo) : 0ull;
    u64 c = (hi << k.vb) | lo;  // vb <= 32, (hi bits + vb) <= 64
    return (u32)(c >> k.shift) & mask;
}

// The same 8-bit digit in 32-bit operations (the branches are uniform): from
// the value half when it lies there, from the key half when it lies there,
// from both when it straddles them.  shift - vb < 32 (the key half has at
// most 32 bits); shift < vb <= 32 otherwise.
__device__ __forceinline__ u32 radix_digit8_hl(u32 hi, u32 lo, const RadixKey &k) {
    if (k.shift >= k.vb) return __builtin_amdgcn_ubfe(hi, k.shift - k.vb, 8);
    u32 d = lo >> k.shift;
    if (k.vb - k.shift < 8) d |= hi << (k.vb - k.shift);
    return d & 0xffu;
}
__device__ __forceinline__ u32 radix_digit8(u64 x, const RadixKey &k) {
    return radix_digit8_hl(tkey(x) - k.min_hi, tval(x) - k.min_lo, k);
}

// min/max of the key and value halves: out[0]=min_hi out[1]=max_hi out[2]=min_lo out[3]=max_lo.
// Each workgroup folds a grid-stride share through the wave and LDS and
// stores its four partials (part[4 b ..]); minmax_final_k folds the
// workgroups' partials.  Device atomics on the four shared words serialised:
// ~100 µs for 2,048 workgroups.
__device__ __forceinline__ void minmax_block(u32 &mnh, u32 &mxh, u32 &mnl, u32 &mxl) {
#pragma unroll
    for (int d = WAVE / 2; d > 0; d >>= 1) {
        mnh = min(mnh, (u32)__shfl_xor((int)mnh, d, WAVE));
        mxh = max(mxh, (u32)__shfl_xor((int)mxh, d, WAVE));
        mnl = min(mnl, (u32)__shfl_xor((int)mnl, d, WAVE));
        mxl = max(mxl, (u32)__shfl_xor((int)mxl, d, WAVE));
    }
    __shared__ u32 sm[4][256 / WAVE];
    const int wave = threadIdx.x / WAVE;
    if ((threadIdx.x & (WAVE - 1)) == 0) {
        sm[0][wave] = mnh; sm[1][wave] = mxh; sm[2][wave] = mnl; sm[3][wave] = mxl;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)(blockDim.x / WAVE); w++) {
            mnh = min(mnh, sm[0][w]); mxh = max(mxh, sm[1][w]);
            mnl = min(mnl, sm[2][w]); mxl = max(mxl, sm[3][w]);
        }
    }
}

__global__ __launch_bounds__(256) void minmax_k(const u64 *in, u64 n, u32 *part) {
    u32 mnh = 0xffffffffu, mxh = 0, mnl = 0xffffffffu, mxl = 0;
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    u64 stride = (u64)gridDim.x * blockDim.x;
    for (; i < n; i += stride) {
        u64 x = in[i];
        u32 h = tkey(x), l = tval(x);
        mnh = min(mnh, h); mxh = max(mxh, h); mnl = min(mnl, l); mxl = max(mxl, l);
    }
    minmax_block(mnh, mxh, mnl, mxl);
    if (threadIdx.x == 0) {
        u32 *p = part + 4 * (u64)blockIdx.x;
        p[0] = mnh; p[1] = mxh; p[2] = mnl; p[3] = mxl;
    }
}

// One workgroup: the fold of nb workgroups' partials (none: the empty bounds).
__global__ __launch_bounds__(256) void minmax_final_k(const u32 *part, u32 nb, u32 *out) {
    u32 mnh = 0xffffffffu, mxh = 0, mnl = 0xffffffffu, mxl = 0;
    for (u32 b = threadIdx.x; b < nb; b += blockDim.x) {
        const u32 *p = part + 4 * (u64)b;
        mnh = min(mnh, p[0]); mxh = max(mxh, p[1]); mnl = min(mnl, p[2]); mxl = max(mxl, p[3]);
    }
    minmax_block(mnh, mxh, mnl, mxl);
    if (threadIdx.x == 0) {
        out[0] = mnh; out[1] = mxh; out[2] = mnl; out[3] = mxl;
    }
}

template <int BITS, int T, int I>
__global__ __launch_bounds__(T) void rs_upsweep_k(const u64 *in, u64 n, RadixKey key, u32 *counts,
                                                  u32 nb) {
    constexpr int BINS = 1 << BITS, W = T / WAVE, TILE = T * I;
    __shared__ u32 h[W][BINS];
    for (int i = threadIdx.x; i < W * BINS; i += T) (&h[0][0])[i] = 0;
    __syncthreads();
    const int wave = threadIdx.x / WAVE;
    u64 base = (u64)blockIdx.x * TILE;
#pragma unroll 4
    for (int r = 0; r < I; r++) {
        u64 idx = base + (u64)r * T + threadIdx.x;
        if (idx < n) atomicAdd(&h[wave][radix_digit(in[idx], key, BINS - 1)], 1u);
    }
    __syncthreads();
    for (int d = threadIdx.x; d < BINS; d += T) {
        u32 s = 0;
#pragma unroll
        for (int w = 0; w < W; w++) s += h[w][d];
        counts[(u64)d * nb + blockIdx.x] = s;
    }
}

// Stable scatter of one tile: wave-match ranking (one ballot per digit bit),
// per-wave running counts in LDS, keys staged in LDS in digit order, then
// written to offs[digit][tile] + rank.  Wave w owns keys
// [tile0 + w*64*I, tile0 + (w+1)*64*I), consumed 64 at a time in order, so
// the (wave, round, lane) order is the input order and the sort is stable.
template <int BITS, int T, int I>
__global__ __launch_bounds__(T) void rs_downsweep_k(const u64 *in, u64 *out, u64 n, RadixKey key,
                                                    const u32 *offs, u32 nb) {
    constexpr int BINS = 1 << BITS, W = T / WAVE, TILE = T * I;
    __shared__ u64 stage[TILE];
    __shared__ u32 wcnt[W][BINS];
    __shared__ u32 bstart[BINS];
    __shared__ u32 gofs[BINS];
    __shared__ u32 sc[T / WAVE + 1];

    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    for (int i = threadIdx.x; i < W * BINS; i += T) (&wcnt[0][0])[i] = 0;
    for (int d = threadIdx.x; d < BINS; d += T) gofs[d] = offs[(u64)d * nb + blockIdx.x];
    __syncthreads();

    const u64 tile0 = (u64)blockIdx.x * TILE;
    const u64 wbase = tile0 + (u64)wave * (WAVE * I);
    const u64 lt = lanemask_lt();
    u64 keys[I];
    u32 pk[I];  // digit | (rank within the wave's digit run << 8)

#pragma unroll
    for (int r = 0; r < I; r++) {
        u64 idx = wbase + (u64)r * WAVE + lane;
        keys[r] = idx < n ? in[idx] : 0ull;
    }
#pragma unroll
    for (int r = 0; r < I; r++) {
        u64 idx = wbase + (u64)r * WAVE + lane;
        bool valid = idx < n;
        u32 d = radix_digit(keys[r], key, BINS - 1);
        u64 m = __ballot(valid);
#pragma unroll
        for (int b = 0; b < BITS; b++) {
            bool bit = (d >> b) & 1u;
            u64 bb = __ballot(bit);
            m &= bit ? bb : ~bb;
        }
        u32 before = __popcll(m & lt);
        u32 cnt = wcnt[wave][d];
        // The lowest lane of each digit group publishes the new running count;
        // every lane of the wave has read the old value in the same LDS op.
        if (valid && before == 0) wcnt[wave][d] = cnt + (u32)__popcll(m);
        pk[r] = d | ((cnt + before) << 8);
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();

    // per digit: exclusive prefix over waves, then over digits
    u32 tot = 0;
    if (threadIdx.x < BINS) {
        u32 s = 0;
#pragma unroll
        for (int w = 0; w < W; w++) {
            u32 c = wcnt[w][threadIdx.x];
            wcnt[w][threadIdx.x] = s;
            s += c;
        }
        tot = s;
    }
    u32 ex = block_exclusive_scan<u32>(tot, sc, nullptr);
    if (threadIdx.x < BINS) bstart[threadIdx.x] = ex;
    __syncthreads();

#pragma unroll
    for (int r = 0; r < I; r++) {
        u64 idx = wbase + (u64)r * WAVE + lane;
        if (idx < n) {
            u32 d = pk[r] & 0xffu;
            stage[bstart[d] + wcnt[wave][d] + (pk[r] >> 8)] = keys[r];
        }
    }
    __syncthreads();

    u64 rem = n - tile0;
    u32 tn = rem < (u64)TILE ? (u32)rem : (u32)TILE;
    for (u32 i = threadIdx.x; i < tn; i += T) {
        u64 x = stage[i];
        u32 d = radix_digit(x, key, BINS - 1);
        out[(u64)gofs[d] + (i - bstart[d])] = x;
    }
}

static int bit_width(u32 v) { return v ? 32 - __builtin_clz(v) : 0; }

template <int BITS, int T, int I>
static u64 *radix_passes(dlg_ctx *ctx, const u64 *src, u64 *dst, u64 *other, u64 n, RadixKey key, int total_bits) {
    constexpr int BINS = 1 << BITS, TILE = T * I;
    u32 nb = (u32)((n + TILE - 1) / TILE);
    DBuf<u32> counts(ctx, (size_t)BINS * nb);
    DBuf<u64> bsum(ctx);
    for (int shift = 0; shift < total_bits; shift += BITS) {
        key.shift = (u32)shift;
        DLG_LAUNCH(ctx, DLG_K_SORT_UPSWEEP, 8.0 * n + 4.0 * BINS * nb, (rs_upsweep_k<BITS, T, I>), nb,
                   T, 0, src, n, key, counts.p, nb);
        scan_u32_inplace(ctx, counts.p, (u64)BINS * nb, bsum);
        DLG_LAUNCH(ctx, DLG_K_SORT_DOWNSWEEP, 16.0 * n + 4.0 * BINS * nb, (rs_downsweep_k<BITS, T, I>),
                   nb, T, 0, src, dst, n, key, (const u32 *)counts.p, nb);
        src = dst;
        std::swap(dst, other);
    }
    return other;
}

// ---------------------------------------------------------- one-sweep passes
// For large inputs with 8-bit digits every pass reads its keys once: one
// histogram kernel counts the digits of all passes in a single read, and
// each pass is one kernel whose tiles take tickets in launch order, rank
// their keys as rs_downsweep_k does, and find where their digit runs go by
// decoupled look-back: a tile publishes its digit counts (AGGREGATE), adds
// the counts of the tiles before it, walking back until a tile that has
// published its inclusive prefix (PREFIX), and publishes its own prefix.  A
// tile only waits for tiles with smaller tickets, which are all running or
// done, so every wait ends; a bounded spin sets an error flag instead of
// hanging should that ever fail.  Status words: tag (8 bits: 2 * pass + 1 for
// AGGREGATE, + 2 for PREFIX, so one zeroed array serves every pass) and
// a 56-bit count.
// Tiles of 512 x 16 keys (64 KiB of LDS staging, two workgroups per CU): on
// 3.4e8 keys 1.82 ms per pass against 2.04 ms for 512 x 32, 2.49 ms for
// 256 x 16 and 1.95-2.53 ms for 256 x 32 (two runs).
constexpr int OS_T = 512, OS_I = 16, OS_TILE = OS_T * OS_I;
constexpr u32 OS_SPIN_LIMIT = 1u << 22;
constexpr u64 OS_VALUE = (1ull << 56) - 1;

// Digits of every pass, counted in one LDS histogram per wave (8 passes x
// 256 bins x 4 waves = 32 KiB), then added into the global counts.  Lanes
// that hit one LDS address in one atomic are serialised, and clustered input
// (sorted runs, hub keys) puts a whole wave on one digit: a wave whose lanes
// share the digit adds its count with one atomic, other waves one per lane.
// A pass whose digits span fewer than 8 bits (the top one) has few distinct
// digits: its count goes through ballot matching, one atomic per distinct
// digit per wave.  Each thread loads OH_I keys of a tile before counting
// any, and the next tile's keys are in flight meanwhile (62 -> 58 us for 10M
// keys).  The kernel is bound by its vector instructions and LDS atomics, so the
// digits come from 32-bit bit-field extracts of the two halves.
constexpr int OH_T = 256, OH_I = 8, OH_TILE = OH_T * OH_I;

__global__ __launch_bounds__(OH_T) void os_hist_k(const u64 *in, u64 n, RadixKey key, u32 passes, u32 top_bits,
                                                  unsigned long long *hist) {
    constexpr int BINS = 256, W = OH_T / WAVE;
    __shared__ u32 h[W][8][BINS];
    for (int i = threadIdx.x; i < W * 8 * BINS; i += OH_T) (&h[0][0][0])[i] = 0;
    __syncthreads();
    const int wave = threadIdx.x / WAVE;
    const u32 p = passes - 1;
    u64 nx[OH_I];   // the next tile's keys, in flight while this one's are counted
    const u64 step = (u64)gridDim.x * OH_TILE;
    {
        const u64 base = (u64)blockIdx.x * OH_TILE;
#pragma unroll
        for (int r = 0; r < OH_I; r++) {
            const u64 i = base + (u64)r * OH_T + threadIdx.x;
            nx[r] = in[i < n ? i : n - 1];
        }
    }
    for (u64 base = (u64)blockIdx.x * OH_TILE; base < n; base += step) {   // block-uniform
        u64 x[OH_I];
#pragma unroll
        for (int r = 0; r < OH_I; r++) x[r] = nx[r];
#pragma unroll
        for (int r = 0; r < OH_I; r++) {   // never predicated: past the end, the last key again (not counted)
            const u64 i = base + step + (u64)r * OH_T + threadIdx.x;
            nx[r] = in[i < n ? i : n - 1];
        }
#pragma unroll
        for (int r = 0; r < OH_I; r++) {
            const bool valid = base + (u64)r * OH_T + threadIdx.x < n;   // valid lanes: a prefix of the wave
            const u64 vm = __ballot(valid);
            if (vm == 0) continue;                                     // wave-uniform
            const u32 hi = tkey(x[r]) - key.min_hi, lo = tval(x[r]) - key.min_lo;
            const u32 nvalid = (u32)__popcll(vm);
            RadixKey kq = key;
            for (u32 q = 0; q < p; q++) {
                kq.shift = 8 * q;
                const u32 dq = radix_digit8_hl(hi, lo, kq);
                const u32 d0 = __builtin_amdgcn_readfirstlane(dq);   // lane 0: valid
                if ((__ballot(dq == d0) & vm) == vm) {
                    if (threadIdx.x % WAVE == 0) atomicAdd(&h[wave][q][d0], nvalid);
                } else if (valid) {
                    atomicAdd(&h[wave][q][dq], 1u);
                }
            }
            kq.shift = 8 * p;
            const u32 d = radix_digit8_hl(hi, lo, kq), nd = ~d;
            u32 mlo = (u32)vm, mhi = (u32)(vm >> 32);
            for (u32 b = 0; b < top_bits; b++) {
                const u32 clr = (u32)__builtin_amdgcn_sbfe((int)nd, b, 1);
                const u64 set = __ballot(clr == 0u);
                mlo &= (u32)set ^ clr;
                mhi &= (u32)(set >> 32) ^ clr;
            }
            const u32 below = __builtin_amdgcn_mbcnt_hi(mhi, __builtin_amdgcn_mbcnt_lo(mlo, 0u));
            if (valid && below == 0) atomicAdd(&h[wave][p][d], (u32)__popc(mlo) + (u32)__popc(mhi));
        }
    }
    __syncthreads();
    for (u32 i = threadIdx.x; i < passes * BINS; i += OH_T) {
        u32 v = 0;   // a workgroup's share of one digit fits 32 bits
#pragma unroll
        for (int w = 0; w < W; w++) v += (&h[w][0][0])[i];
        if (v) atomicAdd(&hist[i], (unsigned long long)v);
    }
}

// Exclusive scan of each pass's digit counts into its digit starts (64-bit:
// one buffer may hold more than 2^32 keys).
__global__ __launch_bounds__(256) void os_starts_k(const u64 *hist, u32 passes, u64 *start) {
    __shared__ u64 sc[256 / WAVE + 1];
    for (u32 p = 0; p < passes; p++) {
        const u64 v = hist[p * 256 + threadIdx.x];
        start[p * 256 + threadIdx.x] = block_exclusive_scan<u64>(v, sc, nullptr);
        __syncthreads();   // sc is reused by the next pass
    }
}

__device__ __forceinline__ u64 os_load(const u64 *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void os_store(u64 *p, u64 v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int T, int I>
__device__ __forceinline__ bool os_load_tile(const u64 *in, u64 n, u64 tile0, u64 wbase, int lane, u64 (&keys)[I]) {
    constexpr int TILE = T * I;
    const bool full = tile0 + TILE <= n;   // every tile but the last: no per-key bounds checks
    if (full) {
#pragma unroll
        for (int r = 0; r < I; r++) keys[r] = in[wbase + (u64)r * WAVE + lane];
    } else {
#pragma unroll
        for (int r = 0; r < I; r++) {
            const u64 idx = wbase + (u64)r * WAVE + lane;
            keys[r] = idx < n ? in[idx] : 0ull;
        }
    }
    return full;
}

template <int T, int I>
__global__ __launch_bounds__(T) void os_pass_k(const u64 *in, u64 *out, u64 n, RadixKey key, const u64 *dstart,
                                               u64 *status, u32 *ticket, u32 pass, u32 *err) {
    constexpr int BINS = 256, W = T / WAVE, TILE = T * I;
    __shared__ u64 stage[TILE];
    __shared__ u32 wcnt[W][BINS];
    __shared__ u32 bstart[BINS];
    __shared__ u64 gofs[BINS];   // output position of stage slot i of digit d: gofs[d] + i (mod 2^64)
    __shared__ u32 sc[T / WAVE + 1];
    __shared__ u32 s_tile;
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    if (threadIdx.x == 0) s_tile = atomicAdd(ticket, 1u);
    for (int i = threadIdx.x; i < W * BINS; i += T) (&wcnt[0][0])[i] = 0;
    __syncthreads();
    const u32 tile = s_tile;
    const u64 tile0 = (u64)tile * TILE;
    const u64 wbase = tile0 + (u64)wave * (WAVE * I);
    u64 keys[I];
    u32 pk[I];   // digit | (rank within the wave's digit run << 8)
    const bool full = os_load_tile<T, I>(in, n, tile0, wbase, lane, keys);
    // Lanes of equal digit by ballot matching: per bit, clr = -1 when the lane's
    // bit is clear, the ballot of clr == 0 is the lanes with it set, and the
    // lane keeps (ballot ^ clr) -- the lanes that agree with it on that bit.
#pragma unroll
    for (int r = 0; r < I; r++) {
        const bool valid = full || wbase + (u64)r * WAVE + lane < n;
        const u32 d = radix_digit8(keys[r], key), nd = ~d;
        const u64 vm = full ? ~0ull : __ballot(valid);
        u32 mlo = (u32)vm, mhi = (u32)(vm >> 32);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const u32 clr = (u32)__builtin_amdgcn_sbfe((int)nd, b, 1);
            const u64 set = __ballot(clr == 0u);
            mlo &= (u32)set ^ clr;
            mhi &= (u32)(set >> 32) ^ clr;
        }
        const u32 before = __builtin_amdgcn_mbcnt_hi(mhi, __builtin_amdgcn_mbcnt_lo(mlo, 0u));
        const u32 cnt = wcnt[wave][d];
        if (valid && before == 0) wcnt[wave][d] = cnt + (u32)__popc(mlo) + (u32)__popc(mhi);
        pk[r] = d | ((cnt + before) << 8);
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    u32 tot = 0;   // the tile's count of digit threadIdx.x; wcnt becomes the exclusive prefix over waves
    if (threadIdx.x < BINS) {
        u32 s = 0;
#pragma unroll
        for (int w = 0; w < W; w++) {
            const u32 c = wcnt[w][threadIdx.x];
            wcnt[w][threadIdx.x] = s;
            s += c;
        }
        tot = s;
    }
    const u32 ex = block_exclusive_scan<u32>(tot, sc, nullptr);
    if (threadIdx.x < BINS) {
        const u32 d = threadIdx.x;
        bstart[d] = ex;
        const u64 agg = (u64)(2 * pass + 1) << 56, pre = (u64)(2 * pass + 2) << 56;
        u64 *mine = status + (u64)tile * BINS + d;
        u64 excl = 0;
        if (tile == 0) {
            os_store(mine, pre | tot);
        } else {
            os_store(mine, agg | tot);
            for (u64 t = tile; t-- > 0;) {
                u64 v = 0;
                for (u32 spin = 0;; spin++) {
                    v = os_load(status + t * BINS + d);
                    const u64 tag = v >> 56;
                    if (tag == 2 * pass + 1 || tag == 2 * pass + 2) break;
                    if (spin >= OS_SPIN_LIMIT) {   // never expected: give up on this digit, flag the sort
                        atomicOr(err, 1u);
                        v = pre;
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                }
                excl += v & OS_VALUE;
                if ((v >> 56) != 2 * pass + 1) break;   // an inclusive prefix (or the flagged give-up)
            }
            os_store(mine, pre | (excl + tot));
        }
        gofs[d] = dstart[d] + excl - (u64)ex;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < I; r++) {
        if (full || wbase + (u64)r * WAVE + lane < n) {
            const u32 d = pk[r] & 0xffu;
            stage[bstart[d] + wcnt[wave][d] + (pk[r] >> 8)] = keys[r];
        }
    }
    __syncthreads();
    const u64 rem = n - tile0;
    const u32 tn = rem < (u64)TILE ? (u32)rem : (u32)TILE;
    for (u32 i = threadIdx.x; i < tn; i += T) {
        const u64 x = stage[i];
        out[gofs[radix_digit8(x, key)] + (u64)i] = x;
    }
}

// All passes of an 8-bit sort: histograms of every pass in one read, then one
// kernel per pass (one read, one write of the keys).
static u64 *radix_onesweep(dlg_ctx *ctx, const u64 *src, u64 *dst, u64 *other, u64 n, RadixKey key, int total_bits) {
    constexpr int OT = OS_T, OI = OS_I, OTILE = OS_TILE;
    const u32 passes = (u32)((total_bits + 7) / 8);
    const u64 tiles = (n + OTILE - 1) / OTILE;
    if (tiles > 0x7fffffffull) fail(DLG_OVERFLOW, "radix sort: too many tiles");
    DBuf<u64> hist(ctx, 8 * 256 * 2);   // histograms, digit starts (64-bit)
    DBuf<u32> tick(ctx, 16);             // tickets, error flag
    DBuf<u64> status(ctx, tiles * 256);
    u64 *starts = hist.p + 8 * 256;
    u32 *tickets = tick.p, *err = tickets + 8;
    fill_u64(ctx, hist.p, 8 * 256 * 2, 0ull);
    fill_u32(ctx, tick.p, 16, 0u);
    fill_u64(ctx, status.p, tiles * 256, 0ull);
    key.shift = 0;
    const u32 top_bits = (u32)(total_bits - 8 * (int)(passes - 1));
    // 4 blocks per CU (32 KiB of LDS each), each looping over tiles
    const unsigned hg = (unsigned)std::min<u64>((n + OH_TILE - 1) / OH_TILE, (u64)ctx->num_cus * 4);
    DLG_LAUNCH(ctx, DLG_K_SORT_UPSWEEP, 8.0 * n, os_hist_k, hg, OH_T, 0, src, n, key, passes, top_bits,
               (unsigned long long *)hist.p);
    DLG_LAUNCH(ctx, DLG_K_SORT_UPSWEEP, 8.0 * 256 * passes, os_starts_k, 1, 256, 0, (const u64 *)hist.p, passes,
               starts);
    for (u32 p = 0; p < passes; p++) {
        key.shift = 8 * p;
        DLG_LAUNCH(ctx, DLG_K_SORT_DOWNSWEEP, 16.0 * n, (os_pass_k<OT, OI>), (unsigned)tiles, OT, 0,
                   src, dst, n, key, (const u64 *)(starts + 256 * p), status.p, tickets + p, p, err);
        src = dst;
        std::swap(dst, other);
    }
    u32 e = 0;
    ctx->read_words(err, 1, &e);
    if (e) fail(DLG_DEVICE_ERROR, "radix sort: a tile's look-back did not complete");
    return other;
}

// The passes from src (left alone) into dst, then between dst and other (which
// may be src); returns the one that holds the sorted keys.
template <int BITS>
static u64 *radix_passes_sized(dlg_ctx *ctx, const u64 *src, u64 *dst, u64 *other, u64 n, RadixKey key, int total_bits) {
    if (BITS == 8 && n >= RS_BIG_MIN) return radix_onesweep(ctx, src, dst, other, n, key, total_bits);
    if (n >= RS_BIG_MIN) return radix_passes<BITS, RS_BIG_T, RS_BIG_I>(ctx, src, dst, other, n, key, total_bits);
    return radix_passes<BITS, RS_SMALL_T, RS_SMALL_I>(ctx, src, dst, other, n, key, total_bits);
}

// ---------------------------------------------------------- sorts by one workgroup
// Up to SS_MAX keys: bounds, every 8-bit pass (ranks as in os_pass_k, keys
// exchanged through LDS) and, as asked, the compaction of the equal runs or the
// key runs' heads, in ONE launch.  Bound by its own latency, about 3 us a pass;
// the launches it replaces (bounds, four a pass, count, scan, scatter) and their
// read-backs took 18 us a pass and about 40 us more: 7,001 tuples of 24 bits 26
// against 95 us, a round of a program's own operators at that size 405 -> 235 us.
// From SORT_SMALL_MAX on, one CU's ranking takes longer than the launches.
constexpr int SS_T = 1024;
enum { SS_SORT = 0, SS_UNIQUE = 1, SS_HEADS = 2 };

// in[0, n) sorted into out (may be in): every tuple (SS_SORT), one of each
// (SS_UNIQUE), or every tuple and the index of each key's first one in heads
// (SS_HEADS); SS_UNIQUE and SS_HEADS publish their count.
template <int I>
__global__ __launch_bounds__(SS_T) void sort_small_k(const u64 *in, u32 n, u64 *out, int mode, int key_only, u32 *heads,
                                                     u64 *host, u64 seq) {
    constexpr int BINS = 256, W = SS_T / WAVE;
    __shared__ u64 stage[SS_T * I];
    __shared__ u32 wcnt[W][BINS];
    __shared__ u32 bstart[BINS];
    __shared__ u32 sc[W + 1];
    __shared__ u32 smm[4][W];
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    const u32 w0 = (u32)wave * (WAVE * I);   // the wave's keys: w0 + r * 64 + lane, in input order
    u64 keys[I];
    u32 mnh = 0xffffffffu, mxh = 0u, mnl = 0xffffffffu, mxl = 0u;
#pragma unroll
    for (int r = 0; r < I; r++) {
        const u32 i = w0 + (u32)r * WAVE + lane;
        keys[r] = i < n ? in[i] : 0ull;
        if (i < n) {
            mnh = min(mnh, tkey(keys[r])); mxh = max(mxh, tkey(keys[r]));
            mnl = min(mnl, tval(keys[r])); mxl = max(mxl, tval(keys[r]));
        }
    }
#pragma unroll
    for (int d = WAVE / 2; d > 0; d >>= 1) {
        mnh = min(mnh, (u32)__shfl_xor((int)mnh, d, WAVE));
        mxh = max(mxh, (u32)__shfl_xor((int)mxh, d, WAVE));
        mnl = min(mnl, (u32)__shfl_xor((int)mnl, d, WAVE));
        mxl = max(mxl, (u32)__shfl_xor((int)mxl, d, WAVE));
    }
    if (lane == 0) {
        smm[0][wave] = mnh; smm[1][wave] = mxh; smm[2][wave] = mnl; smm[3][wave] = mxl;
    }
    __syncthreads();
    for (int w = 0; w < W; w++) {
        mnh = min(mnh, smm[0][w]); mxh = max(mxh, smm[1][w]);
        mnl = min(mnl, smm[2][w]); mxl = max(mxl, smm[3][w]);
    }
    RadixKey key;
    key.min_hi = mnh;
    key.min_lo = mnl;
    key.vb = key_only ? 0u : 32u - (u32)__builtin_clz((mxl - mnl) | 1u) - (mxl == mnl ? 1u : 0u);
    const u32 hb = 32u - (u32)__builtin_clz((mxh - mnh) | 1u) - (mxh == mnh ? 1u : 0u);
    const u32 bits = key.vb + hb;
    for (u32 shift = 0; shift < bits; shift += 8) {   // block-uniform
        key.shift = shift;
        for (int i = threadIdx.x; i < W * BINS; i += SS_T) (&wcnt[0][0])[i] = 0;
        __syncthreads();
        u32 pk[I];
#pragma unroll
        for (int r = 0; r < I; r++) {
            const bool valid = w0 + (u32)r * WAVE + lane < n;
            const u32 d = radix_digit8(keys[r], key), nd = ~d;
            const u64 vm = __ballot(valid);
            u32 mlo = (u32)vm, mhi = (u32)(vm >> 32);
#pragma unroll
            for (int b = 0; b < 8; b++) {
                const u32 clr = (u32)__builtin_amdgcn_sbfe((int)nd, b, 1);
                const u64 set = __ballot(clr == 0u);
                mlo &= (u32)set ^ clr;
                mhi &= (u32)(set >> 32) ^ clr;
            }
            const u32 before = __builtin_amdgcn_mbcnt_hi(mhi, __builtin_amdgcn_mbcnt_lo(mlo, 0u));
            const u32 cnt = wcnt[wave][d];
            if (valid && before == 0) wcnt[wave][d] = cnt + (u32)__popc(mlo) + (u32)__popc(mhi);
            pk[r] = d | ((cnt + before) << 8);
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();
        u32 tot = 0;
        if (threadIdx.x < BINS) {
#pragma unroll
            for (int w = 0; w < W; w++) {
                const u32 c = wcnt[w][threadIdx.x];
                wcnt[w][threadIdx.x] = tot;
                tot += c;
            }
        }
        const u32 ex = block_exclusive_scan<u32>(tot, sc, nullptr);
        if (threadIdx.x < BINS) bstart[threadIdx.x] = ex;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < I; r++)
            if (w0 + (u32)r * WAVE + lane < n) {
                const u32 d = pk[r] & 0xffu;
                stage[bstart[d] + wcnt[wave][d] + (pk[r] >> 8)] = keys[r];
            }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < I; r++) {
            const u32 i = w0 + (u32)r * WAVE + lane;
            if (i < n) keys[r] = stage[i];
        }
    }
    if (bits == 0) {   // all equal (or sorted by a key they share): as they came
#pragma unroll
        for (int r = 0; r < I; r++) {
            const u32 i = w0 + (u32)r * WAVE + lane;
            if (i < n) stage[i] = keys[r];
        }
        __syncthreads();
    }
    if (mode != SS_UNIQUE) {
#pragma unroll
        for (int r = 0; r < I; r++) {
            const u32 i = w0 + (u32)r * WAVE + lane;
            if (i < n) out[i] = keys[r];
        }
        if (mode == SS_SORT) return;
    }
    u32 keep = 0;
#pragma unroll
    for (int r = 0; r < I; r++) {   // each thread's I consecutive tuples
        const u32 i = threadIdx.x * I + r;
        if (i < n && (i == 0 || (mode == SS_HEADS ? tkey(stage[i]) != tkey(stage[i - 1]) : stage[i] != stage[i - 1])))
            keep |= 1u << r;
    }
    u32 total;
    u32 at = block_exclusive_scan<u32>((u32)__popc(keep), sc, &total);
#pragma unroll
    for (int r = 0; r < I; r++)
        if ((keep >> r) & 1u) {
            const u32 i = threadIdx.x * I + r;
            if (mode == SS_HEADS) heads[at++] = i;
            else out[at++] = stage[i];
        }
    if (threadIdx.x == 0) {
        host[0] = total;
        __threadfence_system();
        *(volatile u64 *)(host + dlg_ctx::MAPPED_SEQ) = seq;
        __threadfence_system();
    }
}

static u64 sort_small(dlg_ctx *ctx, const u64 *in, u64 n, u64 *out, int mode, bool key_only, u32 *heads) {
    const u64 seq = mode == SS_SORT ? 0 : ++ctx->mapped_seq;
    auto go = [&](auto kern) {
        DLG_LAUNCH(ctx, DLG_K_SORT_DOWNSWEEP, 16.0 * n, kern, 1, SS_T, 0, in, (u32)n, out, mode, key_only ? 1 : 0, heads,
                   ctx->mapped_dev(seq), seq);
    };
    if (n <= SS_T) go(sort_small_k<1>);
    else if (n <= 2 * SS_T) go(sort_small_k<2>);
    else if (n <= 4 * SS_T) go(sort_small_k<4>);
    else go(sort_small_k<8>);
    if (mode == SS_SORT) return n;
    ctx->wait_mapped(seq);
    return ((const volatile u64 *)ctx->mapped_host(seq))[0];
}

u64 sort_unique_small(dlg_ctx *ctx, const u64 *in, u64 n, u64 *out) {
    return sort_small(ctx, in, n, out, SS_UNIQUE, false, nullptr);
}
u64 sort_heads_small(dlg_ctx *ctx, const u64 *in, u64 n, u64 *out, u32 *heads) {
    return sort_small(ctx, in, n, out, SS_HEADS, false, heads);
}

// The bounds of a few tuples, one launch that publishes them (a fold by workgroups, one of their
// partials and a read-back otherwise).
__global__ __launch_bounds__(SS_T) void minmax_small_k(const u64 *data, u32 n, u64 *host, u64 seq) {
    u32 b[4] = {0xffffffffu, 0u, 0xffffffffu, 0u};
    for (u32 i = threadIdx.x; i < n; i += SS_T) {
        const u64 x = data[i];
        b[0] = min(b[0], tkey(x)); b[1] = max(b[1], tkey(x));
        b[2] = min(b[2], tval(x)); b[3] = max(b[3], tval(x));
    }
    __shared__ u32 sm[4][SS_T / WAVE];
#pragma unroll
    for (int q = 0; q < 4; q++) {
#pragma unroll
        for (int d = WAVE / 2; d > 0; d >>= 1) {
            const u32 o = (u32)__shfl_xor((int)b[q], d, WAVE);
            b[q] = q & 1 ? max(b[q], o) : min(b[q], o);
        }
        if (threadIdx.x % WAVE == 0) sm[q][threadIdx.x / WAVE] = b[q];
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int w = 1; w < SS_T / WAVE; w++)
        for (int q = 0; q < 4; q++) b[q] = q & 1 ? max(b[q], sm[q][w]) : min(b[q], sm[q][w]);
    host[0] = (u64)b[1] << 32 | b[0];
    host[1] = (u64)b[3] << 32 | b[2];
    __threadfence_system();
    *(volatile u64 *)(host + dlg_ctx::MAPPED_SEQ) = seq;
    __threadfence_system();
}

void tuple_bounds(dlg_ctx *ctx, const u64 *data, u64 n, u32 *h) {
    if (n <= SORT_SMALL_MAX) {
        const u64 seq = ++ctx->mapped_seq;
        DLG_LAUNCH(ctx, DLG_K_SORT_HIST, 8.0 * n, minmax_small_k, 1, SS_T, 0, data, (u32)n, ctx->mapped_dev(seq), seq);
        ctx->wait_mapped(seq);
        std::memcpy(h, (const void *)ctx->mapped_host(seq), 16);
        return;
    }
    const unsigned g = n ? (unsigned)std::min<u64>((n + 255) / 256, (u64)ctx->num_cus * 8) : 0u;
    DBuf<u32> mm(ctx, 4 + 4 * (u64)g);   // the bounds, then the workgroups' partials
    if (g) DLG_LAUNCH(ctx, DLG_K_SORT_HIST, 8.0 * n, minmax_k, g, 256, 0, data, n, mm.p + 4);
    DLG_LAUNCH(ctx, DLG_K_MISC, 16.0 * g, minmax_final_k, 1, 256, 0, (const u32 *)(mm.p + 4), g, mm.p);
    ctx->read_words(mm.p, 4, h);
}

// Per block: the digest sum and the order breaks of a grid-stride share,
// reduced through the wave and LDS, then one atomic each.
// A tuple's terms of the digest, the constants' products taken out: the sums of
// r0, r1 and r0 r1 give sum(r0 C0 + r1 C1 + r0 r1 + C2) mod 2^64 at the end, so a
// tuple costs one multiplication.
struct RdSum {
    u64 s0 = 0, s1 = 0, p = 0;
    __device__ __forceinline__ void add(u64 t, int orient) {
        const u32 k = tkey(t) ^ 0x80000000u, v = tval(t) ^ 0x80000000u;   // the int32 bits
        s0 += orient == DLG_ORIENT_KV ? k : v;
        s1 += orient == DLG_ORIENT_KV ? v : k;
        p += (u64)k * v;
    }
    __device__ __forceinline__ u64 total() const { return s0 * 0x9E3779B97F4A7C15ull + s1 * 0xC2B2AE3D27D4EB4Full + p; }
};

// d[0, 2 np): RD_U pairs a thread in flight, 16 bytes each (d is 16-byte aligned;
// kernel takes a tuple before and after them alone).  Bound by the one read: 2.0e9
// tuples 3.45 -> 2.85 ms (5.7 TB/s) against a tuple a thread with three products;
// 2 and 4 pairs in flight 3.01 and 2.91.
constexpr int RD_T = 256, RD_U = 8;
__global__ __launch_bounds__(RD_T) void rows_digest_k(const u64 *d, u64 n, int orient, unsigned long long *acc) {
    __shared__ u64 s_sum[RD_T / WAVE], s_brk[RD_T / WAVE];
    const u64 np = n / 2;
    RdSum sum;
    u64 brk = 0, consts = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        consts = n * 0x632BE59BD9B4E019ull;
        if (n & 1) sum.add(d[n - 1], orient);
    }
    const u64 stride = (u64)gridDim.x * RD_T * RD_U;
    for (u64 base = (u64)blockIdx.x * RD_T * RD_U; base < np; base += stride) {   // block-uniform
        ulonglong2 t[RD_U];
        u64 nx[RD_U];
#pragma unroll
        for (int u = 0; u < RD_U; u++) {   // past the end: the last pair again, not counted
            const u64 i = min(base + (u64)u * RD_T + threadIdx.x, np - 1);
            t[u] = *(const ulonglong2 *)(d + 2 * i);
            nx[u] = d[min(2 * i + 2, n - 1)];   // past the last pair: its second tuple, or the one after it
        }
#pragma unroll
        for (int u = 0; u < RD_U; u++) {
            const u64 i = base + (u64)u * RD_T + threadIdx.x;
            if (i < np) {
                sum.add(t[u].x, orient);
                sum.add(t[u].y, orient);
                brk += t[u].x >= t[u].y;
                brk += 2 * i + 2 < n && t[u].y >= nx[u];
            }
        }
    }
    u64 v = sum.total() + consts;
#pragma unroll
    for (int o = WAVE / 2; o > 0; o >>= 1) {
        v += __shfl_xor(v, o, WAVE);
        brk += __shfl_xor(brk, o, WAVE);
    }
    const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
    if (lane == 0) {
        s_sum[w] = v;
        s_brk[w] = brk;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int j = 1; j < RD_T / WAVE; j++) {
            v += s_sum[j];
            brk += s_brk[j];
        }
        atomicAdd(acc, (unsigned long long)v);
        atomicAdd(acc + 1, (unsigned long long)brk);
    }
}

void rows_digest(dlg_ctx *ctx, const u64 *d, u64 n, int orient, u64 *sum, u64 *breaks) {
    if ((size_t)d & 15u) fail(DLG_INVALID_INPUT, "rows_digest: unaligned tuples");   // a pool block's start
    DBuf<u64> acc(ctx, 2);
    fill_u64(ctx, acc.p, 2, 0ull);
    if (n) {
        unsigned g = (unsigned)std::min<u64>((n + 2 * RD_T * RD_U - 1) / (2 * RD_T * RD_U), (u64)ctx->num_cus * 8);
        DLG_LAUNCH(ctx, DLG_K_MISC, 8.0 * n, rows_digest_k, g, RD_T, 0, d, n, orient,
                   (unsigned long long *)acc.p);
    }
    u64 h[2];
    ctx->read_scalars(acc.p, 2, h);
    *sum = h[0];
    *breaks = h[1];
}

// in[0, n) sorted into a or b (b may be in): returns the one that holds the
// result -- `in` itself when there is nothing to do.
static const u64 *radix_from(dlg_ctx *ctx, const u64 *in, u64 n, u64 *a, u64 *b, int bits, const u32 *bounds, bool key_only) {
    if (n < 2) return in;
    if (n <= SORT_SMALL_MAX) {
        sort_small(ctx, in, n, b, SS_SORT, key_only, nullptr);
        return b;
    }
    if (bits <= 0) bits = ctx->radix_bits;
    if (bits < 4) bits = 4;
    if (bits > 8) bits = 8;
    // The 8-bit onesweep counts digits in 64 bits; the narrower digit passes
    // keep 32-bit digit offsets.
    if (n > 0xffffffffull && bits != 8)
        fail(DLG_OVERFLOW, "radix_sort: more than 2^32-1 tuples need 8-bit digits");
    u32 h[4];
    if (bounds) std::memcpy(h, bounds, sizeof(h));
    else tuple_bounds(ctx, in, n, h);
    RadixKey key;
    key.min_hi = h[0];
    key.min_lo = h[2];
    key.vb = key_only ? 0u : (u32)bit_width(h[3] - h[2]);   // key_only: a stable sort by key alone
    key.shift = 0;
    int total_bits = (int)key.vb + bit_width(h[1] - h[0]);
    if (total_bits == 0) return in;  // all equal
    switch (bits) {
        case 4: return radix_passes_sized<4>(ctx, in, a, b, n, key, total_bits);
        case 5: return radix_passes_sized<5>(ctx, in, a, b, n, key, total_bits);
        case 6: return radix_passes_sized<6>(ctx, in, a, b, n, key, total_bits);
        case 7: return radix_passes_sized<7>(ctx, in, a, b, n, key, total_bits);
        default: return radix_passes_sized<8>(ctx, in, a, b, n, key, total_bits);
    }
}

void radix_sort(dlg_ctx *ctx, DBuf<u64> &data, u64 n, DBuf<u64> &tmp, int bits, const u32 *bounds,
                bool key_only) {
    if (n < 2) return;
    if (n > SORT_SMALL_MAX) tmp.ensure(n);   // the one-workgroup sort works in place
    const u64 *r = radix_from(ctx, data.p, n, tmp.p, data.p, bits, bounds, key_only);
    if (r != data.p) data.swap(tmp);   // result is in the other buffer: swap ownership
}

void radix_sort_into(dlg_ctx *ctx, const u64 *in, u64 n, DBuf<u64> &out, DBuf<u64> &tmp) {
    out.ensure(n ? n : 1);
    if (n > SORT_SMALL_MAX) tmp.ensure(n);
    const u64 *r = radix_from(ctx, in, n, tmp.p, out.p, 0, nullptr, false);
    if (r == in) copy_u64(ctx, out.p, in, n);
    else if (r != out.p) out.swap(tmp);
}

void radix_sort(dlg_ctx *ctx, u64 *data, u64 n, DBuf<u64> &tmp, int bits, bool key_only) {
    if (n < 2) return;
    if (n > SORT_SMALL_MAX) tmp.ensure(n);
    const u64 *r = radix_from(ctx, data, n, tmp.p, data, bits, nullptr, key_only);
    if (r != data) copy_u64(ctx, data, r, n);   // sorted copy ended in tmp; bring it back
}

u64 sort_unique(dlg_ctx *ctx, u64 *data, u64 n) {
    if (n == 0) return 0;
    if (n <= SORT_SMALL_MAX) return sort_unique_small(ctx, data, n, data);
    DBuf<u64> tmp(ctx, n);
    const u64 *r = radix_from(ctx, data, n, tmp.p, data, 0, nullptr, false);
    if (r != data) return select(ctx, SEL_UNIQUE, r, n, nullptr, 0, data);   // compacted straight back
    const u64 k = select(ctx, SEL_UNIQUE, data, n, nullptr, 0, tmp.p);
    copy_u64(ctx, data, tmp.p, k);
    return k;
}

// =============================================================== select
constexpr int SEL_T = 256, SEL_I = 8, SEL_TILE = SEL_T * SEL_I;

__device__ __forceinline__ bool found_sorted(const u64 *a, u64 lo, u64 hi, u64 x) {
    u64 p = lower_bound_u64(a, lo, hi, x);
    return p < hi && a[p] == x;
}

template <int MODE>
__global__ __launch_bounds__(SEL_T) void select_count_k(const u64 *in, u64 n, u64 *flags, u64 *bsum) {
    __shared__ u64 sc[SEL_T / WAVE + 1];
    const u64 base = (u64)blockIdx.x * SEL_TILE;
    u64 c = 0;
#pragma unroll
    for (int r = 0; r < SEL_I; r++) {
        u64 idx = base + (u64)r * SEL_T + threadIdx.x;
        bool keep = false;
        if (idx < n) {
            u64 x = in[idx];
            if (MODE == SEL_KEY_HEAD) {
                keep = idx == 0 || tkey(in[idx - 1]) != tkey(x);
            } else if (MODE == SEL_NODIAG) {
                keep = tkey(x) != tval(x);
            } else {
                keep = idx == 0 || in[idx - 1] != x;
                if (MODE == SEL_UNIQUE_NODIAG) keep = keep && tkey(x) != tval(x);
            }
        }
        u64 m = __ballot(keep);
        u64 w0 = base + (u64)r * SEL_T + (threadIdx.x & ~(WAVE - 1));
        if ((threadIdx.x & (WAVE - 1)) == 0 && w0 < n) flags[w0 / WAVE] = m;
        c += keep ? 1 : 0;
    }
    u64 tot;
    block_exclusive_scan<u64>(c, sc, &tot);
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// The same flags for the modes that drop what sorted `other` holds (UNIQUE:
// equal runs too).  The tile goes by SEL_PARTS parts; a part's stretch of
// `other` begins at split[part] (select_split_k) and, up to SEL_STAGE elements,
// comes into LDS with coalesced reads (all of them in flight together) and is
// searched there; a larger one is searched in global memory.
// 16M elements against 33M: 86 us (4.6 TB/s) against 291 us with every search in
// global memory, each tile's range found by a wave; 176 us with the staging's
// loads one after the other.
constexpr int SEL_PARTS = 4, SEL_PART = SEL_TILE / SEL_PARTS, SEL_PER = SEL_I / SEL_PARTS;
constexpr u32 SEL_BATCH = 8;
constexpr u64 SEL_STAGE = SEL_BATCH * SEL_T;

// split[p] = the first of `other` not below in[p SEL_PART], and, past the last
// part, the first above in[n - 1]: one thread each (a wave's 64 pivots per step
// would read 64 lines per search).
__global__ __launch_bounds__(256) void select_split_k(const u64 *in, u64 n, const u64 *other, u64 no, u64 parts, u64 *split) {
    const u64 p = (u64)blockIdx.x * 256 + threadIdx.x;
    if (p < parts) split[p] = lower_bound_u64(other, 0, no, in[p * SEL_PART]);
    else if (p == parts) split[p] = upper_bound_u64(other, 0, no, in[n - 1]);
}

template <bool UNIQUE>
__global__ __launch_bounds__(SEL_T) void select_minus_k(const u64 *in, u64 n, const u64 *other, const u64 *split, u64 parts,
                                                        u64 *flags, u64 *bsum) {
    __shared__ u64 s_other[SEL_STAGE];
    __shared__ u64 sc[SEL_T / WAVE + 1];
    const u64 base = (u64)blockIdx.x * SEL_TILE;
    u64 c = 0;
    for (int part = 0; part < SEL_PARTS; part++) {
        const u64 p = (u64)blockIdx.x * SEL_PARTS + part;
        if (p >= parts) break;   // block-uniform
        const u64 lo = split[p];
        // the next part's first element may be this part's last one too
        const u64 hi = split[p + 1] + (p + 1 < parts && split[p + 1] < split[parts] ? 1 : 0);
        const bool staged = hi - lo <= SEL_STAGE;
        const u64 i0 = base + (u64)part * SEL_PART + threadIdx.x;
        u64 x[SEL_PER], before[SEL_PER];
#pragma unroll
        for (int r = 0; r < SEL_PER; r++) {
            const u64 i = i0 + (u64)r * SEL_T;
            x[r] = i < n ? in[i] : 0ull;
            if (UNIQUE) before[r] = i > 0 && i < n ? in[i - 1] : 0ull;
        }
        const u32 m = (u32)(hi - lo);
        if (staged && m) {
            u64 v[SEL_BATCH];
#pragma unroll
            for (u32 k = 0; k < SEL_BATCH; k++)
                if (k * SEL_T < m) v[k] = other[lo + min(k * SEL_T + threadIdx.x, m - 1)];   // uniform
#pragma unroll
            for (u32 k = 0; k < SEL_BATCH; k++)
                if (k * SEL_T < m) s_other[k * SEL_T + threadIdx.x] = v[k];
        }
        __syncthreads();
        bool found[SEL_PER];
        if (staged) {
            u32 at[SEL_PER];
#pragma unroll
            for (int r = 0; r < SEL_PER; r++) at[r] = 0;
            for (u32 len = m; len > 1; len -= len / 2) {   // block-uniform: the searches step together
                const u32 half = len / 2;
                u64 v[SEL_PER];
#pragma unroll
                for (int r = 0; r < SEL_PER; r++) v[r] = s_other[at[r] + half - 1];
#pragma unroll
                for (int r = 0; r < SEL_PER; r++) at[r] += v[r] < x[r] ? half : 0u;
            }
#pragma unroll
            for (int r = 0; r < SEL_PER; r++) found[r] = m && s_other[at[r]] == x[r];
        } else {
#pragma unroll
            for (int r = 0; r < SEL_PER; r++) found[r] = found_sorted(other, lo, hi, x[r]);
        }
#pragma unroll
        for (int r = 0; r < SEL_PER; r++) {
            const u64 i = i0 + (u64)r * SEL_T;
            const bool keep = i < n && !found[r] && (!UNIQUE || i == 0 || before[r] != x[r]);
            const u64 bal = __ballot(keep);
            const u64 w0 = i & ~(u64)(WAVE - 1);
            if ((threadIdx.x & (WAVE - 1)) == 0 && w0 < n) flags[w0 / WAVE] = bal;
            c += keep;
        }
        __syncthreads();   // the stretch is searched: the next part's comes in
    }
    u64 tot;
    block_exclusive_scan<u64>(c, sc, &tot);
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

template <bool OUT_INDEX>
__global__ __launch_bounds__(SEL_T) void select_scatter_k(const u64 *in, u64 n, const u64 *flags,
                                                          const u64 *bpre, void *out) {
    __shared__ u32 wc[SEL_I][SEL_T / WAVE];
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    const u64 base = (u64)blockIdx.x * SEL_TILE;
    u64 words[SEL_I];
#pragma unroll
    for (int r = 0; r < SEL_I; r++) {
        u64 w0 = base + (u64)r * SEL_T + (u64)wave * WAVE;
        words[r] = w0 < n ? flags[w0 / WAVE] : 0ull;
        if (lane == 0) wc[r][wave] = (u32)__popcll(words[r]);
    }
    __syncthreads();
    u64 pre = bpre[blockIdx.x];
    const u64 lt = lanemask_lt();
#pragma unroll
    for (int r = 0; r < SEL_I; r++) {
        u32 p = 0;
        for (int rr = 0; rr < SEL_I; rr++)
            for (int ww = 0; ww < SEL_T / WAVE; ww++)
                if (rr < r || (rr == r && ww < wave)) p += wc[rr][ww];
        if ((words[r] >> lane) & 1ull) {
            u64 idx = base + (u64)r * SEL_T + threadIdx.x;
            u64 pos = pre + p + (u64)__popcll(words[r] & lt);
            if (OUT_INDEX) ((u32 *)out)[pos] = (u32)idx;
            else ((u64 *)out)[pos] = in[idx];
        }
    }
}

// The whole compaction by one workgroup, for up to SORT_SMALL_MAX elements:
// flags, scan, scatter and the count's publication in one launch.  A thread
// takes 8 consecutive elements; its searches of `other` step together.
template <int MODE>
__global__ __launch_bounds__(1024) void select_small_k(const u64 *in, u32 n, const u64 *other, u64 no, void *out, u64 *host,
                                                       u64 seq) {
    constexpr int I = (int)(SORT_SMALL_MAX / 1024);
    constexpr bool NEED_OTHER = (MODE == SEL_UNIQUE_NOT_IN || MODE == SEL_NOT_IN);
    __shared__ u64 s_piv[NEED_OTHER ? 1024 : 1];
    __shared__ u32 sc[1024 / WAVE + 1];
    const u64 stride = (no + 1023) / 1024;   // `other` in 1024 segments, their last elements in LDS
    if (NEED_OTHER) {
        const u64 e = ((u64)threadIdx.x + 1) * stride;
        s_piv[threadIdx.x] = other[(e < no ? e : no) - 1];
        __syncthreads();
    }
    const u32 i0 = threadIdx.x * I;
    u64 x[I];
#pragma unroll
    for (int r = 0; r < I; r++) x[r] = i0 + r < n ? in[i0 + r] : 0ull;
    const u64 before = i0 > 0 && i0 < n ? in[i0 - 1] : 0ull;
    u32 keep = 0;
#pragma unroll
    for (int r = 0; r < I; r++) {
        if (i0 + r >= n) continue;
        const u64 prev = r ? x[r ? r - 1 : 0] : before;
        const bool first = i0 + r == 0;
        bool k = true;
        if (MODE == SEL_KEY_HEAD) k = first || tkey(prev) != tkey(x[r]);
        else if (MODE == SEL_UNIQUE || MODE == SEL_UNIQUE_NODIAG || MODE == SEL_UNIQUE_NOT_IN) k = first || prev != x[r];
        if (MODE == SEL_UNIQUE_NODIAG || MODE == SEL_NODIAG) k = k && tkey(x[r]) != tval(x[r]);
        keep |= k ? 1u << r : 0u;
    }
    if (NEED_OTHER) {
        // each element's segment among the pivots in LDS, then its place in the
        // segment: log2(no / 1024) dependent reads of global memory instead of log2(no)
        u64 lo[I];
#pragma unroll
        for (int r = 0; r < I; r++) {
            u32 a = 0;   // pivots below x
#pragma unroll
            for (u32 h = 512; h; h >>= 1) a += s_piv[a + h - 1] < x[r] ? h : 0u;
            lo[r] = (u64)a * stride;   // the last pivot below x may be the last of all: then x is in no segment
        }
        for (u64 len = stride; len > 1; len -= len / 2) {   // block-uniform: the searches step together
            const u64 half = len / 2;
            u64 v[I];
#pragma unroll
            for (int r = 0; r < I; r++) v[r] = lo[r] + half - 1 < no ? other[lo[r] + half - 1] : ~0ull;
#pragma unroll
            for (int r = 0; r < I; r++) lo[r] += v[r] < x[r] ? half : 0;
        }
#pragma unroll
        for (int r = 0; r < I; r++)
            if (lo[r] < no && other[lo[r]] == x[r]) keep &= ~(1u << r);
    }
    u32 total;
    u32 at = block_exclusive_scan<u32>((u32)__popc(keep), sc, &total);   // every read is done before the first write
#pragma unroll
    for (int r = 0; r < I; r++)
        if ((keep >> r) & 1u) {
            if (MODE == SEL_KEY_HEAD) ((u32 *)out)[at++] = i0 + r;
            else ((u64 *)out)[at++] = x[r];
        }
    if (threadIdx.x == 0) {
        host[0] = total;
        __threadfence_system();
        *(volatile u64 *)(host + dlg_ctx::MAPPED_SEQ) = seq;
        __threadfence_system();
    }
}

template <int MODE>
static u64 select_small(dlg_ctx *ctx, const u64 *in, u64 n, const u64 *other, u64 n_other, void *out) {
    const u64 seq = ++ctx->mapped_seq;
    DLG_LAUNCH(ctx, DLG_K_SELECT, 16.0 * n, select_small_k<MODE>, 1, 1024, 0, in, (u32)n, other, n_other, out,
               ctx->mapped_dev(seq), seq);
    ctx->wait_mapped(seq);
    return ((const volatile u64 *)ctx->mapped_host(seq))[0];
}

// The positions of the set bits among `n` flags: a thread takes a word, as few are
// set (select_scatter_k has a thread a row: 2.6e8 rows with 4.9M heads 252 us, most of it
// its 128,000 workgroups; 20 here).  bpre: the bits before each workgroup's words.
constexpr u64 HW_ROWS = (u64)SEL_T * WAVE;   // rows a workgroup
constexpr u64 HW_SPARSE = 8;                 // rows a head from which on
__global__ __launch_bounds__(SEL_T) void heads_sum_k(const u64 *flags, u64 words, u64 *bsum) {
    __shared__ u64 sc[SEL_T / WAVE + 1];
    const u64 w = (u64)blockIdx.x * SEL_T + threadIdx.x;
    u64 tot;
    block_exclusive_scan<u64>(w < words ? (u64)__popcll(flags[w]) : 0ull, sc, &tot);
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}
__global__ __launch_bounds__(SEL_T) void heads_scatter_k(const u64 *flags, u64 words, const u64 *bpre, u64 step, u32 *out) {
    __shared__ u64 sc[SEL_T / WAVE + 1];
    const u64 w = (u64)blockIdx.x * SEL_T + threadIdx.x;
    const u64 f = w < words ? flags[w] : 0ull;
    u64 at = block_exclusive_scan<u64>((u64)__popcll(f), sc, nullptr) + bpre[blockIdx.x * step];
    for (u64 b = f; b; b &= b - 1) out[at++] = (u32)(w * WAVE + (u64)__ffsll((unsigned long long)b) - 1);
}
u64 select_flagged(dlg_ctx *ctx, const u64 *flags, u64 n, u32 *out) {
    if (n == 0) return 0;
    const u64 words = (n + WAVE - 1) / WAVE, nb = (n + HW_ROWS - 1) / HW_ROWS;
    DBuf<u64> bsum(ctx, nb), tot(ctx, 1);
    DLG_LAUNCH(ctx, DLG_K_SELECT, 8.0 * words, heads_sum_k, (unsigned)nb, SEL_T, 0, flags, words, bsum.p);
    scan_blocks(ctx, bsum.p, nb, tot.p);
    u64 total = 0;
    ctx->read_scalars(tot.p, 1, &total);
    DLG_LAUNCH(ctx, DLG_K_SELECT, 8.0 * words + 4.0 * total, heads_scatter_k, (unsigned)nb, SEL_T, 0, flags, words,
               (const u64 *)bsum.p, 1ull, out);
    return total;
}

u64 select(dlg_ctx *ctx, int mode, const u64 *in, u64 n, const u64 *other, u64 n_other,
           void *out) {
    if (n == 0) return 0;
    if ((mode == SEL_NOT_IN || mode == SEL_UNIQUE_NOT_IN) && n_other == 0)
        mode = mode == SEL_NOT_IN ? -1 : SEL_UNIQUE;
    if (mode == -1) {  // nothing to remove
        if (out != (const void *)in) copy_u64(ctx, (u64 *)out, in, n);
        return n;
    }
    if (n <= SORT_SMALL_MAX) switch (mode) {
        case SEL_UNIQUE: return select_small<SEL_UNIQUE>(ctx, in, n, other, n_other, out);
        case SEL_UNIQUE_NODIAG: return select_small<SEL_UNIQUE_NODIAG>(ctx, in, n, other, n_other, out);
        case SEL_UNIQUE_NOT_IN: return select_small<SEL_UNIQUE_NOT_IN>(ctx, in, n, other, n_other, out);
        case SEL_NOT_IN: return select_small<SEL_NOT_IN>(ctx, in, n, other, n_other, out);
        case SEL_KEY_HEAD: return select_small<SEL_KEY_HEAD>(ctx, in, n, other, n_other, out);
        case SEL_NODIAG: return select_small<SEL_NODIAG>(ctx, in, n, other, n_other, out);
        default: fail(DLG_INVALID_INPUT, "select: bad mode");
    }
    u64 nb = (n + SEL_TILE - 1) / SEL_TILE;
    DBuf<u64> flags(ctx, (n + WAVE - 1) / WAVE + 1);
    DBuf<u64> bsum(ctx, nb);
    DBuf<u64> tot(ctx, 1);
    const double rb = 8.0 * n + 8.0 * ((n + 63) / 64);
    if (mode == SEL_NOT_IN || mode == SEL_UNIQUE_NOT_IN) {
        const u64 parts = (n + SEL_PART - 1) / SEL_PART;
        DBuf<u64> split(ctx, parts + 1);
        DLG_LAUNCH(ctx, DLG_K_SELECT, 16.0 * parts, select_split_k, grid_for(parts + 1, 256), 256, 0, in, n, other, n_other,
                   parts, split.p);
        if (mode == SEL_NOT_IN)
            DLG_LAUNCH(ctx, DLG_K_SELECT, rb + 8.0 * n_other, select_minus_k<false>, (unsigned)nb, SEL_T, 0, in, n, other,
                       (const u64 *)split.p, parts, flags.p, bsum.p);
        else
            DLG_LAUNCH(ctx, DLG_K_SELECT, rb + 8.0 * n_other, select_minus_k<true>, (unsigned)nb, SEL_T, 0, in, n, other,
                       (const u64 *)split.p, parts, flags.p, bsum.p);
    } else {
        auto go = [&](auto kern) {
            DLG_LAUNCH(ctx, DLG_K_SELECT, rb, kern, (unsigned)nb, SEL_T, 0, in, n, flags.p, bsum.p);
        };
        switch (mode) {
            case SEL_UNIQUE: go(select_count_k<SEL_UNIQUE>); break;
            case SEL_UNIQUE_NODIAG: go(select_count_k<SEL_UNIQUE_NODIAG>); break;
            case SEL_KEY_HEAD: go(select_count_k<SEL_KEY_HEAD>); break;
            case SEL_NODIAG: go(select_count_k<SEL_NODIAG>); break;
            default: fail(DLG_INVALID_INPUT, "select: bad mode");
        }
    }
    scan_blocks(ctx, bsum.p, nb, tot.p);
    u64 total = 0;
    ctx->read_scalars(tot.p, 1, &total);
    if (total == 0) return 0;
    if (mode == SEL_KEY_HEAD && total <= n / HW_SPARSE)
        DLG_LAUNCH(ctx, DLG_K_SELECT, 8.0 * ((n + 63) / 64) + 4.0 * total, heads_scatter_k, (unsigned)((n + HW_ROWS - 1) / HW_ROWS),
                   SEL_T, 0, (const u64 *)flags.p, (n + WAVE - 1) / WAVE, (const u64 *)bsum.p, HW_ROWS / SEL_TILE, (u32 *)out);
    else if (mode == SEL_KEY_HEAD)
        DLG_LAUNCH(ctx, DLG_K_SELECT, 8.0 * ((n + 63) / 64) + 12.0 * total,
                   select_scatter_k<true>, (unsigned)nb, SEL_T, 0, in, n, flags.p, bsum.p, out);
    else
        DLG_LAUNCH(ctx, DLG_K_SELECT, 8.0 * ((n + 63) / 64) + 16.0 * total,
                   select_scatter_k<false>, (unsigned)nb, SEL_T, 0, in, n, flags.p, bsum.p, out);
    return total;
}

// First of each equal run of sorted `in` and absent from every run of `rs`.
// Each block narrows every run to the range spanned by its own tile (one
// thread per run), so a candidate's searches stay inside small ranges.
__global__ __launch_bounds__(SEL_T) void select_count_runs_k(const u64 *in, u64 n, RunSet rs,
                                                             u64 *flags, u64 *bsum) {
    __shared__ u64 s_lo[MAX_RUNS], s_hi[MAX_RUNS];
    __shared__ u64 sc[SEL_T / WAVE + 1];
    const u64 base = (u64)blockIdx.x * SEL_TILE;
    if ((int)threadIdx.x < rs.k) {
        const int j = threadIdx.x;
        u64 last = base + SEL_TILE - 1 < n ? base + SEL_TILE - 1 : n - 1;
        u64 lo = lower_bound_u64(rs.p[j], 0, rs.n[j], in[base]);
        s_lo[j] = lo;
        s_hi[j] = upper_bound_u64(rs.p[j], lo, rs.n[j], in[last]);
    }
    __syncthreads();
    u64 c = 0;
#pragma unroll
    for (int r = 0; r < SEL_I; r++) {
        u64 idx = base + (u64)r * SEL_T + threadIdx.x;
        bool keep = false;
        if (idx < n) {
            u64 x = in[idx];
            keep = idx == 0 || in[idx - 1] != x;
            for (int j = 0; keep && j < rs.k; j++)
                if (s_lo[j] < s_hi[j]) keep = !found_sorted(rs.p[j], s_lo[j], s_hi[j], x);
        }
        u64 m = __ballot(keep);
        u64 w0 = base + (u64)r * SEL_T + (threadIdx.x & ~(WAVE - 1));
        if ((threadIdx.x & (WAVE - 1)) == 0 && w0 < n) flags[w0 / WAVE] = m;
        c += keep ? 1 : 0;
    }
    u64 tot;
    block_exclusive_scan<u64>(c, sc, &tot);
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

u64 select_unique_not_in_runs(dlg_ctx *ctx, const u64 *in, u64 n, const RunSet &rs, u64 *out) {
    if (n == 0) return 0;
    if (rs.k == 0) return select(ctx, SEL_UNIQUE, in, n, nullptr, 0, out);
    u64 nb = (n + SEL_TILE - 1) / SEL_TILE;
    DBuf<u64> flags(ctx, (n + WAVE - 1) / WAVE + 1);
    DBuf<u64> bsum(ctx, nb);
    DBuf<u64> tot(ctx, 1);
    DLG_LAUNCH(ctx, DLG_K_SELECT, 8.0 * n + 8.0 * ((n + 63) / 64), select_count_runs_k,
               (unsigned)nb, SEL_T, 0, in, n, rs, flags.p, bsum.p);
    scan_blocks(ctx, bsum.p, nb, tot.p);
    u64 total = 0;
    ctx->read_scalars(tot.p, 1, &total);
    if (total == 0) return 0;
    DLG_LAUNCH(ctx, DLG_K_SELECT, 8.0 * ((n + 63) / 64) + 16.0 * total, select_scatter_k<false>,
               (unsigned)nb, SEL_T, 0, in, n, flags.p, bsum.p, (void *)out);
    return total;
}

// =============================================================== merge
// Merge path: output tile t of MP_TILE elements takes a[split[t], split[t+1])
// and the matching stretch of b; the split of diagonal d is the number of
// a-elements among the first d outputs of the stable merge (a first on ties).
constexpr int MP_T = 256, MP_I = 8, MP_TILE = MP_T * MP_I, MP_SPLIT_T = 256;

// One thread per diagonal d = t * MP_TILE, t in [0, tiles]: a plain binary search
// (a wave's 64 pivots per step would read 64 lines per step for every diagonal).
__global__ __launch_bounds__(MP_SPLIT_T) void merge_split_k(const u64 *a, u64 na, const u64 *b, u64 nb,
                                                            u64 tiles, u64 *split) {
    const u64 t = (u64)blockIdx.x * MP_SPLIT_T + threadIdx.x;
    if (t > tiles) return;
    const u64 n = na + nb, d = t * MP_TILE < n ? t * MP_TILE : n;
    u64 lo = d > nb ? d - nb : 0, hi = d < na ? d : na;
    while (lo < hi) {   // a[m] > b[d-1-m] turns true at the split; d-1-m stays in [0, nb)
        const u64 m = (lo + hi) >> 1;
        if (a[m] > b[d - 1 - m]) hi = m; else lo = m + 1;
    }
    split[t] = lo;
}

// Tile blockIdx.x of the merge: a's stretch and b's side by side in s, then
// this thread's MP_I outputs (tile positions [t MP_I, t MP_I + MP_I), valid
// below the returned count) merged into v.  s is still being read when it
// returns: a barrier must come before s is written again.
__device__ __forceinline__ int mp_tile(const u64 *a, u64 na, const u64 *b, u64 nb, const u64 *split, u64 *s,
                                       u64 (&v)[MP_I]) {
    const u64 n = na + nb, d0 = (u64)blockIdx.x * MP_TILE;
    const int cnt = (int)(n - d0 < (u64)MP_TILE ? n - d0 : (u64)MP_TILE);
    const u64 i0 = split[blockIdx.x], j0 = d0 - i0;
    const int ca = (int)(split[blockIdx.x + 1] - i0), cb = cnt - ca;
#pragma unroll
    for (int r = 0; r < MP_I; r++) {
        const int k = r * MP_T + (int)threadIdx.x;
        if (k < cnt) s[k] = k < ca ? a[i0 + (u64)k] : b[j0 + (u64)(k - ca)];
    }
    __syncthreads();
    const int dt = (int)threadIdx.x * MP_I;
    if (dt < cnt) {
        int lo = dt > cb ? dt - cb : 0, hi = dt < ca ? dt : ca;
        while (lo < hi) {   // this thread's split inside the tile
            const int m = (lo + hi) >> 1;
            if (s[m] <= s[ca + dt - 1 - m]) lo = m + 1; else hi = m;
        }
        int ia = lo, ib = dt - lo;
        u64 va = ia < ca ? s[ia] : 0, vb = ib < cb ? s[ca + ib] : 0;
#pragma unroll
        for (int r = 0; r < MP_I; r++) {
            const bool take_a = ia < ca && (ib >= cb || va <= vb);
            v[r] = take_a ? va : vb;
            if (take_a) {
                ia++;
                va = ia < ca ? s[ia] : 0;
            } else {
                ib++;
                vb = ib < cb ? s[ca + ib] : 0;
            }
        }
    }
    return cnt;
}

__global__ __launch_bounds__(MP_T) void merge_path_k(const u64 *a, u64 na, const u64 *b, u64 nb,
                                                     const u64 *split, u64 *out) {
    __shared__ u64 s[MP_TILE];
    u64 v[MP_I];
    const int cnt = mp_tile(a, na, b, nb, split, s, v);
    const int dt = (int)threadIdx.x * MP_I;
    __syncthreads();
    if (dt < cnt) {
#pragma unroll
        for (int r = 0; r < MP_I; r++)
            if (dt + r < cnt) s[dt + r] = v[r];
    }
    __syncthreads();
    const u64 d0 = (u64)blockIdx.x * MP_TILE;
#pragma unroll
    for (int r = 0; r < MP_I; r++) {
        const int k = r * MP_T + (int)threadIdx.x;
        if (k < cnt) out[d0 + (u64)k] = s[k];
    }
}

// Merge keeping one copy of each value: an output is kept when it differs
// from the one before it (the tile's first compares with the element before
// the tile: the larger of a[i0 - 1] and b[j0 - 1]).  Pass 1 (SCATTER false)
// writes each tile's count to tcnt; pass 2 reads the tiles' exclusive
// offsets there, compacts the kept outputs in LDS and stores them coalesced.
template <bool SCATTER>
__global__ __launch_bounds__(MP_T) void merge_unique_k(const u64 *a, u64 na, const u64 *b, u64 nb,
                                                       const u64 *split, u64 *tcnt, u64 *out) {
    __shared__ u64 s[MP_TILE];
    __shared__ u64 s_last[MP_T];
    __shared__ u64 sc[MP_T / WAVE + 1];
    u64 v[MP_I];
    const int cnt = mp_tile(a, na, b, nb, split, s, v);
    const int dt = (int)threadIdx.x * MP_I;
    const int m = dt < cnt ? (cnt - dt < MP_I ? cnt - dt : MP_I) : 0;   // this thread's valid outputs
    if (m) s_last[threadIdx.x] = v[m - 1];
    u64 prev = 0;
    bool has_prev = threadIdx.x > 0;
    if (threadIdx.x == 0 && blockIdx.x > 0) {   // the element before the tile
        const u64 i0 = split[blockIdx.x], j0 = (u64)blockIdx.x * MP_TILE - i0;
        const u64 pa = i0 ? a[i0 - 1] : 0, pb = j0 ? b[j0 - 1] : 0;
        prev = pa > pb ? pa : pb;
        has_prev = true;
    }
    __syncthreads();
    if (threadIdx.x > 0) prev = s_last[threadIdx.x - 1];   // a thread with outputs follows a full one
    u32 keep = 0, nk = 0;
#pragma unroll
    for (int r = 0; r < MP_I; r++) {
        if (r < m) {
            const bool k = !has_prev || v[r] != prev;
            keep |= (u32)k << r;
            nk += k;
            prev = v[r];
            has_prev = true;
        }
    }
    u64 tot;
    u64 pos = block_exclusive_scan<u64>(nk, sc, &tot);   // its barriers also end the tile's reads of s
    if (!SCATTER) {
        if (threadIdx.x == 0) tcnt[blockIdx.x] = tot;
        return;
    }
#pragma unroll
    for (int r = 0; r < MP_I; r++)
        if ((keep >> r) & 1u) s[pos++] = v[r];
    __syncthreads();
    const u64 o0 = tcnt[blockIdx.x];
    for (u64 k = threadIdx.x; k < tot; k += MP_T) out[o0 + k] = s[k];
}

static u64 merge_splits(dlg_ctx *ctx, const u64 *a, u64 na, const u64 *b, u64 nb, DBuf<u64> &split) {
    const u64 tiles = (na + nb + MP_TILE - 1) / MP_TILE;
    split.ensure(tiles + 1);
    DLG_LAUNCH(ctx, DLG_K_MERGE, 16.0 * (tiles + 1), merge_split_k, grid_for(tiles + 1, MP_SPLIT_T), MP_SPLIT_T, 0,
               a, na, b, nb, tiles, split.p);
    return tiles;
}

void merge(dlg_ctx *ctx, const u64 *a, u64 na, const u64 *b, u64 nb, u64 *out) {
    const u64 n = na + nb;
    if (n == 0) return;
    DBuf<u64> split(ctx);
    const u64 tiles = merge_splits(ctx, a, na, b, nb, split);
    DLG_LAUNCH(ctx, DLG_K_MERGE, 16.0 * n, merge_path_k, (unsigned)tiles, MP_T, 0, a, na, b, nb,
               (const u64 *)split.p, out);
}

u64 merge_unique(dlg_ctx *ctx, const u64 *a, u64 na, const u64 *b, u64 nb, u64 *out) {
    const u64 n = na + nb;
    if (n == 0) return 0;
    DBuf<u64> split(ctx), tcnt(ctx), tot(ctx, 1);
    const u64 tiles = merge_splits(ctx, a, na, b, nb, split);
    tcnt.ensure(tiles);
    DLG_LAUNCH(ctx, DLG_K_MERGE, 8.0 * n, merge_unique_k<false>, (unsigned)tiles, MP_T, 0, a, na, b, nb,
               (const u64 *)split.p, tcnt.p, (u64 *)nullptr);
    scan_blocks(ctx, tcnt.p, tiles, tot.p);
    u64 total = 0;
    ctx->read_scalars(tot.p, 1, &total);
    if (total == 0) return 0;
    DLG_LAUNCH(ctx, DLG_K_MERGE, 8.0 * n + 8.0 * total, merge_unique_k<true>, (unsigned)tiles, MP_T, 0, a, na, b,
               nb, (const u64 *)split.p, tcnt.p, out);
    return total;
}

}  // namespace dlg
