// libpercolate_hip: MI355X (gfx950, wave64, CDNA4) kernels for the
// Newman-Ziff bond-percolation hot path, behind the C ABI declared in
// include/percolate_hip.h.
//
// Pipeline for R runs on a graph with N nodes and M edges:
//   permute (Philox-keyed bucket shuffle, or MT19937 + numpy's shuffle for
//   bit-exact RandomState permutations) -> sweep (union-find: square
//   lattices in tiles, one wavefront per run and tile, then the events
//   between tiles; other graphs one run per workgroup of one or two
//   wavefronts; merge records) -> chunk states
//   (per-run state every 64
//   steps: two passes over the records, or written by the sweep itself) ->
//   microcanonical sums (exact Sigma x, Sigma x^2 over runs per step) or
//   expand (per-run traces) -> canonical averages (binomial convolution on
//   the matrix cores, the weights generated inside the contraction).
//
// The observables of one run at step s (largest cluster, spanning flag,
// moments k = 0..4 of all clusters but the largest) depend only on the set
// of bonds occupied after s steps.  With Sk(s) = sum over all clusters of
// size**k they are exact prefix functions of the merge records (a, b):
//   max(s) = max(1, max over merges <= s of a + b)
//   #clusters(s) = N - merges(s)
//   Sk(s) = N + sum over merges <= s of (a + b)**k - a**k - b**k
//   moments_k(s) = Sk(s) - max(s)**k      (k = 0: #clusters - 1)
// which equals the reference's incremental bookkeeping
// (percolate/hpc.py:282-305) whichever largest cluster it excludes on ties.
#include <hip/hip_runtime.h>

#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <type_traits>
#include <vector>

#include "percolate_hip.h"
#include "stirlerr_table.h"

typedef unsigned __int128 u128;

// ---------------------------------------------------------------------------
// Error reporting
// ---------------------------------------------------------------------------
static thread_local char g_last_error[512];

static int pc_fail(int code, const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_last_error, sizeof g_last_error, fmt, ap);
    va_end(ap);
    return code;
}

#define PC_HIP_CHECK(expr)                                                     \
    do {                                                                       \
        hipError_t e_ = (expr);                                                \
        if (e_ != hipSuccess)                                                  \
            return pc_fail(PC_EHIP, "%s failed: %s", #expr,                    \
                           hipGetErrorString(e_));                             \
    } while (0)

#define PC_LAUNCH_CHECK(name)                                                  \
    do {                                                                       \
        hipError_t e_ = hipGetLastError();                                     \
        if (e_ != hipSuccess)                                                  \
            return pc_fail(PC_EHIP, "launch of %s failed: %s", name,           \
                           hipGetErrorString(e_));                             \
    } while (0)

// ---------------------------------------------------------------------------
// Wavefront helpers (wave64).  Scans use DPP row shifts inside each row of
// 16 lanes and the GFX9 row broadcasts 15 / 31 across rows.
// ---------------------------------------------------------------------------
#define DPP_ROW_SHR(n) (0x110 + (n))
#define DPP_ROW_BCAST15 0x142
#define DPP_ROW_BCAST31 0x143

template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ uint32_t dpp32(uint32_t v)
{
    // lanes without a source (row edge or masked row) read 0, the identity
    // of every scan below (sum and unsigned max)
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK,
                                                 0xf, false);
}

template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ uint64_t dpp64(uint64_t v)
{
    return (uint64_t)dpp32<CTRL, ROW_MASK>((uint32_t)v) |
           ((uint64_t)dpp32<CTRL, ROW_MASK>((uint32_t)(v >> 32)) << 32);
}

template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ u128 dpp128(u128 v)
{
    return (u128)dpp64<CTRL, ROW_MASK>((uint64_t)v) |
           ((u128)dpp64<CTRL, ROW_MASK>((uint64_t)(v >> 64)) << 64);
}

template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ uint32_t dpp_any(uint32_t v) { return dpp32<CTRL, ROW_MASK>(v); }
template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ uint64_t dpp_any(uint64_t v) { return dpp64<CTRL, ROW_MASK>(v); }
template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ u128 dpp_any(u128 v) { return dpp128<CTRL, ROW_MASK>(v); }

// Inclusive prefix sum over the 64 lanes.
template <typename T>
__device__ __forceinline__ T wave_scan_add(T x)
{
    x += dpp_any<DPP_ROW_SHR(1)>(x);
    x += dpp_any<DPP_ROW_SHR(2)>(x);
    x += dpp_any<DPP_ROW_SHR(4)>(x);
    x += dpp_any<DPP_ROW_SHR(8)>(x);
    x += dpp_any<DPP_ROW_BCAST15, 0xa>(x);
    x += dpp_any<DPP_ROW_BCAST31, 0xc>(x);
    return x;
}

// Inclusive prefix scans over the 64 lanes of a chunk's state in one go: the
// maximum mx and the sums d2, d3, d4 (32 to 128 bits), in place with DPP adds
// and carries (one instruction per word and step; the scans' steps alternate,
// so no step waits for its own previous result).  Row shifts read 0 past a
// row's edge; the two row broadcasts leave the rows they do not add to as they
// are.  Against separate scans of moved copies: 26, 48 and 60 instructions
// per chunk and step of the sums instead of 80 to 170.
#define SCAN_SHR(n) "row_shr:" #n " row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
#define SCAN_B15 "row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
#define SCAN_B31 "row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
#define SCAN_MAX(r, c) "v_max_u32_dpp " r ", " r ", " r " " c
#define SCAN_ADD(r, c) "v_add_u32_dpp " r ", " r ", " r " " c
#define SCAN_ADD_CO(r, c) "v_add_co_u32_dpp " r ", vcc, " r ", " r " " c
#define SCAN_ADDC(r, c) "v_addc_co_u32_dpp " r ", vcc, " r ", " r ", vcc " c
#define SCAN_64(lo, hi, c) SCAN_ADD_CO(lo, c) SCAN_ADDC(hi, c)
#define SCAN_128(a, b, d, e, c) SCAN_ADD_CO(a, c) SCAN_ADDC(b, c) SCAN_ADDC(d, c) SCAN_ADDC(e, c)
#define SCAN_STEPS(S) S(SCAN_SHR(1)) S(SCAN_SHR(2)) S(SCAN_SHR(4)) S(SCAN_SHR(8)) S(SCAN_B15) S(SCAN_B31)
// sums over the rows of 16 lanes alone: the total in a row's last lane
#define SCAN_ROWS(S) S(SCAN_SHR(1)) S(SCAN_SHR(2)) S(SCAN_SHR(4)) S(SCAN_SHR(8))
// wait states between the compiler's write of an operand and the first DPP
// read, and between the last write and a lane read
#define SCAN_NOP "s_nop 1\n\t"

#define SCAN_STEP_NARROW(c) SCAN_MAX("%0", c) SCAN_ADD("%1", c) SCAN_64("%2", "%3", c) SCAN_64("%4", "%5", c)
#define SCAN_96(a, b, d, c) SCAN_ADD_CO(a, c) SCAN_ADDC(b, c) SCAN_ADDC(d, c)
#define SCAN_STEP_96(c) SCAN_MAX("%0", c) SCAN_64("%1", "%2", c) SCAN_64("%3", "%4", c) SCAN_96("%5", "%6", "%7", c)
#define SCAN_STEP_WIDE(c) SCAN_MAX("%0", c) SCAN_64("%1", "%2", c) SCAN_128("%3", "%4", "%5", "%6", c) SCAN_128("%7", "%8", "%9", "%10", c)

typedef unsigned _BitInt(96) u96;

struct Words128 {
    uint32_t w[4];
    __device__ __forceinline__ explicit Words128(u128 v)
        : w{(uint32_t)v, (uint32_t)(v >> 32), (uint32_t)(v >> 64), (uint32_t)(v >> 96)} {}
    __device__ __forceinline__ u128 value() const
    {
        return ((u128)(((uint64_t)w[3] << 32) | w[2]) << 64) | (((uint64_t)w[1] << 32) | w[0]);
    }
};

#define SCAN_DEFINE(NAME, STEPS)                                                           \
    __device__ __forceinline__ void NAME(uint32_t &mx, uint32_t &d2, uint64_t &d3,         \
                                         uint64_t &d4)                                     \
    {                                                                                      \
        uint32_t a = (uint32_t)d3, b = (uint32_t)(d3 >> 32);                               \
        uint32_t c = (uint32_t)d4, d = (uint32_t)(d4 >> 32);                               \
        asm volatile(SCAN_NOP STEPS(SCAN_STEP_NARROW) SCAN_NOP                             \
                     : "+v"(mx), "+v"(d2), "+v"(a), "+v"(b), "+v"(c), "+v"(d)::"vcc");     \
        d3 = ((uint64_t)b << 32) | a;                                                      \
        d4 = ((uint64_t)d << 32) | c;                                                      \
    }                                                                                      \
    __device__ __forceinline__ void NAME(uint32_t &mx, uint64_t &d2, uint64_t &d3,         \
                                         u96 &d4)                                          \
    {                                                                                      \
        uint32_t a = (uint32_t)d2, b = (uint32_t)(d2 >> 32);                               \
        uint32_t c = (uint32_t)d3, d = (uint32_t)(d3 >> 32);                               \
        uint32_t e = (uint32_t)d4, f = (uint32_t)(d4 >> 32), g = (uint32_t)(d4 >> 64);     \
        asm volatile(SCAN_NOP STEPS(SCAN_STEP_96) SCAN_NOP                                 \
                     : "+v"(mx), "+v"(a), "+v"(b), "+v"(c), "+v"(d), "+v"(e), "+v"(f),     \
                       "+v"(g)::"vcc");                                                    \
        d2 = ((uint64_t)b << 32) | a;                                                      \
        d3 = ((uint64_t)d << 32) | c;                                                      \
        d4 = ((u96)g << 64) | ((u96)f << 32) | e;                                          \
    }                                                                                      \
    __device__ __forceinline__ void NAME(uint32_t &mx, uint64_t &d2, u128 &d3, u128 &d4)   \
    {                                                                                      \
        uint32_t a = (uint32_t)d2, b = (uint32_t)(d2 >> 32);                               \
        Words128 c(d3), e(d4);                                                             \
        asm volatile(SCAN_NOP STEPS(SCAN_STEP_WIDE) SCAN_NOP                               \
                     : "+v"(mx), "+v"(a), "+v"(b), "+v"(c.w[0]), "+v"(c.w[1]),             \
                       "+v"(c.w[2]), "+v"(c.w[3]), "+v"(e.w[0]), "+v"(e.w[1]),             \
                       "+v"(e.w[2]), "+v"(e.w[3])::"vcc");                                 \
        d2 = ((uint64_t)b << 32) | a;                                                      \
        d3 = c.value();                                                                    \
        d4 = e.value();                                                                    \
    }
SCAN_DEFINE(scan_state, SCAN_STEPS)
SCAN_DEFINE(scan_state_rows, SCAN_ROWS)

// The lanes of the mask below this one.
__device__ __forceinline__ uint32_t lanes_below(uint64_t mask)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                     __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// Lanes up to and including this one with the flag set.
__device__ __forceinline__ uint32_t scan_count(bool flag)
{
    return lanes_below(__ballot(flag)) + (flag ? 1u : 0u);
}

__device__ __forceinline__ uint64_t umax64(uint64_t a, uint64_t b) { return a > b ? a : b; }

// Lanes whose flag is set.  (__ballot compares the flag, widened to a
// register, with 0: two vector instructions that a lane mask does not need.)
__device__ __forceinline__ uint64_t ballot(bool flag) { return __builtin_amdgcn_ballot_w64(flag); }

// The first active lane's value, as a wave-uniform (scalar) value.
__device__ __forceinline__ uint32_t uniform(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}


__device__ __forceinline__ uint32_t read_lane(uint32_t v, uint32_t lane)
{
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)lane);
}
__device__ __forceinline__ uint64_t read_lane(uint64_t v, uint32_t lane)
{
    return (uint64_t)read_lane((uint32_t)v, lane) |
           ((uint64_t)read_lane((uint32_t)(v >> 32), lane) << 32);
}
__device__ __forceinline__ u128 read_lane(u128 v, uint32_t lane)
{
    return (u128)read_lane((uint64_t)v, lane) |
           ((u128)read_lane((uint64_t)(v >> 64), lane) << 64);
}

// Multi-word atomic adds: each word's carry-out is recovered from the old
// value the atomic returns, so concurrent adders compose exactly.
__device__ __forceinline__ void atomic_add_u128(uint64_t *p, u128 v)
{
    uint64_t lo = (uint64_t)v, hi = (uint64_t)(v >> 64);
    if (lo) {
        unsigned long long old = atomicAdd((unsigned long long *)p, lo);
        if (old + lo < old)
            hi += 1;
    }
    if (hi)
        atomicAdd((unsigned long long *)(p + 1), hi);
}

__device__ __forceinline__ void atomic_add_u192(uint64_t *p, uint64_t w0,
                                                uint64_t w1, uint64_t w2)
{
    if (w0) {
        unsigned long long old = atomicAdd((unsigned long long *)p, w0);
        if (old + w0 < old) {
            w1 += 1;
            if (w1 == 0)
                w2 += 1;
        }
    }
    if (w1) {
        unsigned long long old = atomicAdd((unsigned long long *)(p + 1), w1);
        if (old + w1 < old)
            w2 += 1;
    }
    if (w2)
        atomicAdd((unsigned long long *)(p + 2), w2);
}

// ---------------------------------------------------------------------------
// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11), the counter-based
// generator of the device permutations.
// ---------------------------------------------------------------------------
struct u32x4 {
    uint32_t x, y, z, w;
};

__device__ __forceinline__ u32x4 philox4x32_10(u32x4 c, uint32_t k0,
                                               uint32_t k1)
{
#pragma unroll
    for (int i = 0; i < 10; ++i) {
        if (i) {
            k0 += 0x9E3779B9u;
            k1 += 0xBB67AE85u;
        }
        const uint64_t p0 = (uint64_t)0xD2511F53u * c.x;
        const uint64_t p1 = (uint64_t)0xCD9E8D57u * c.z;
        c = u32x4{(uint32_t)(p1 >> 32) ^ c.y ^ k0, (uint32_t)p1,
                  (uint32_t)(p0 >> 32) ^ c.w ^ k1, (uint32_t)p0};
    }
    return c;
}

// ---------------------------------------------------------------------------
// Device permutations (performance mode): a Rao-Sandelius shuffle keyed by
// Philox4x32-10.  Every element draws a uniform random bucket label; the
// elements are grouped by label in a stable counting sort (one radix pass
// over random keys), and every bucket is shuffled uniformly: a second level
// of random labels, then Fisher-Yates with unbiased bounded draws inside
// each sub-bucket.  With independent uniform words the result is an exactly
// uniform permutation: iid labels plus a uniform order inside each label
// class is a sort by iid continuous keys.
//
// Layout (the oracle's nz_shuffle.c restates it; perm[i] = edge index added
// at step i + 1):
//   - M <= SHUF_WHOLE: the whole run is one bucket (lb1 = 0), shuffled by
//     one workgroup straight from the identity.  Otherwise 2^lb1 buckets,
//     lb1 the least with M <= SHUF_BUCKET << lb1; label of element i = the
//     top lb1 bits of key(1, 0, i).
//   - Bucket b of n elements, in their grouped (increasing) order: in runs
//     of several buckets, n > SHUF_GROUP_CAP (odds below e^-1500 at these
//     sizes): plain Fisher-Yates in HBM with 32-bit draws from ctr
//     (u, run, b, 4 << 28).  Otherwise
//     2^lb2 sub-buckets (the least lb2 with n <= SHUF_SUB << lb2), label of
//     position j = the top lb2 bits of key(2, b, j), stable grouping, then
//     Fisher-Yates of each sub-bucket (start st, size c) with 16-bit draws:
//     the halves of ctr (st, run, b, 3 << 28 | u) in turn, a rejected word
//     replaced by the next half of ctr (st, run, b, 5 << 28 | v).  Every
//     accepted draw so takes exactly one word of the first stream, and the
//     lanes of a wave, which start their sub-buckets together, refill it
//     together.
//   - key(tag, b, j) = 16-bit half (j >> 6) & 7 (low half first) of
//     Philox(ctr ((j >> 9) << 6 | (j & 63), run, b, tag << 28)): one Philox
//     call per lane labels 8 positions 64 apart, so a wave labels 512
//     consecutive positions per call and visits them in order.
//   - Bounded draw on [0, r) from a w-bit word x: m = x * r, rejected while
//     (m mod 2^w) < (2^w - r) mod r (Lemire), result m >> w.
// Kernels: for several buckets count (labels per bucket and chunk of
// SHUF_CHUNK elements) -> scan (per run) -> scatter (stable grouping into
// the output row); then group (one workgroup per bucket, in LDS).
// ---------------------------------------------------------------------------
#define SHUF_BUCKET 4096u
#define SHUF_GROUP_CAP 8192u
#define SHUF_WHOLE 32768u
#define SHUF_SUB 64u
#define SHUF_SMALL_CAP 4096u  // one-bucket runs up to this size: 2-wave groups
#define SHUF_CHUNK 4096u
#define SHUF_MAX_EDGES (1u << 23)
#define SHUF_W 4

__device__ __forceinline__ uint32_t half16(const u32x4 &w, uint32_t h)
{
    const uint32_t wd = (h & 4u) ? ((h & 2u) ? w.w : w.z) : ((h & 2u) ? w.y : w.x);
    return (wd >> ((h & 1u) * 16u)) & 0xFFFFu;
}

__device__ __forceinline__ u32x4 shuf_philox(uint32_t x, uint32_t run, uint32_t b,
                                             uint32_t w, uint32_t k0, uint32_t k1)
{
    return philox4x32_10(u32x4{x, run, b, w}, k0, k1);
}

// Lanes (of the active ones in `valid`) whose label equals this lane's, for a
// label of `bits` bits: one ballot per bit.  Per bit, s is all ones where
// the lane's bit is set, and each 32-bit half of the mask keeps the lanes
// whose ballot bit equals s (one three-input bit operation per half).
__device__ __forceinline__ uint64_t match_label(uint32_t label, uint32_t bits,
                                                uint64_t valid)
{
    uint32_t lo = (uint32_t)valid, hi = (uint32_t)(valid >> 32);
    for (uint32_t i = 0; i < bits; ++i) {
        const uint32_t s = (uint32_t)((int32_t)(label << (31u - i)) >> 31);
        const uint64_t ones = ballot(s != 0u);
        lo &= ~((uint32_t)ones ^ s);
        hi &= ~((uint32_t)(ones >> 32) ^ s);
    }
    return ((uint64_t)hi << 32) | lo;
}

// match_label through LDS: every lane sets its bit in the mask of its label's
// low `in_lds` bits, a table of the wave's own (all zero before and after),
// and reads the mask back; only the bits above cost a ballot, of four vector
// instructions each.  Lanes outside `ok` get no peers.  The kernels that group
// by label are bound by vector issue (80 to 92 % busy with a ballot for each
// of 7 to 9 bits), so this pays: grouping by 512 labels, 2.1e9 edges, 7.1 ms
// with ballots and labels drawn twice, 5.0; whole runs of 32512 edges (10^4)
// 1.17 ms, 0.97 (5, 6 and 8 bits here: 1.08, 1.03 and 1.32: a table of 8 bits
// leaves room for fewer workgroups, one of few bits has lanes wait for each
// other).  shuf_match_bits says where fewer bits pay.
#define MATCH_BITS 7u
#define MATCH_WORDS (2u << MATCH_BITS)   // 32-bit words of a wave's table

__device__ __forceinline__ uint64_t match_label_lds(uint32_t label, uint32_t bits,
                                                    bool ok, unsigned long long *table,
                                                    uint32_t in_lds = MATCH_BITS)
{
    unsigned long long *slot = table + (label & ((1u << in_lds) - 1u));
    uint64_t peers = 0;
    if (ok) {
        __hip_atomic_fetch_or(slot, 1ull << (threadIdx.x & 63u), __ATOMIC_RELAXED,
                              __HIP_MEMORY_SCOPE_WORKGROUP);
        peers = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __hip_atomic_store(slot, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    return bits > in_lds ? match_label(label >> in_lds, bits - in_lds, peers) : peers;
}

// Lemire's rejection threshold (2^w - r) mod r for w = 16 and w = 32, called
// only when a draw's low part is below r.  The empty asm hides r from the
// optimiser, which would otherwise hoist the integer division out of the
// rare branch and pay it on every draw.
__device__ __forceinline__ uint32_t lemire_threshold16(uint32_t r)
{
    asm volatile("" : "+v"(r));
    return (65536u - r) % r;
}
__device__ __forceinline__ uint32_t lemire_threshold32(uint32_t r)
{
    asm volatile("" : "+v"(r));
    return (0u - r) % r;
}

// A rejected 16-bit draw (m = x * r with m mod 2^16 < r) redrawn from the
// sub-bucket's replacement stream until accepted; v counts the replacement
// words taken.
__device__ __forceinline__ uint32_t shuffle_redraw(uint32_t m, uint32_t r,
                                                   uint32_t st, uint32_t run,
                                                   uint32_t b, uint32_t k0,
                                                   uint32_t k1, uint32_t &v)
{
    const uint32_t thr = lemire_threshold16(r);
    while ((m & 0xFFFFu) < thr) {
        const u32x4 w = shuf_philox(st, run, b, (5u << 28) | (v >> 3), k0, k1);
        const uint32_t h = v & 7u;
        const uint32_t wd = (h & 4u) ? ((h & 2u) ? w.w : w.z) : ((h & 2u) ? w.y : w.x);
        m = ((wd >> ((h & 1u) * 16u)) & 0xFFFFu) * r;
        ++v;
    }
    return m;
}

// Fisher-Yates of a[0..c) with the 16-bit draw streams of sub-bucket start
// st.  The Philox words are kept as scalars: a struct indexed by the running
// half counter would be demoted to a private (scratch or LDS) array.
template <typename E>
__device__ __forceinline__ void shuffle_sub(E *a, uint32_t c, uint32_t st,
                                            uint32_t run, uint32_t b, uint32_t k0,
                                            uint32_t k1)
{
    uint32_t v = 0u;
    // eight draws a Philox call
    for (uint32_t j0 = c - 1u, u = 0u; (int32_t)j0 >= 1; j0 -= 8u, ++u) {
        const u32x4 w = shuf_philox(st, run, b, (3u << 28) | u, k0, k1);
#pragma unroll
        for (uint32_t h = 0; h < 8u; ++h) {
            const uint32_t j = j0 - h, r = j + 1u;
            if ((int32_t)j < 1)
                break;
            // 16-bit word times r <= 2^15 + 1: a 24-bit multiply is exact
            uint32_t m = __umul24(half16(w, h), r);
            if (__builtin_expect((m & 0xFFFFu) < r, 0))
                m = shuffle_redraw(m, r, st, run, b, k0, k1, v);
            const uint32_t k = m >> 16;
            const E t = a[j];
            a[j] = a[k];
            a[k] = t;
        }
    }
}

// Fisher-Yates of a bucket of n > SHUF_GROUP_CAP elements in HBM, 32-bit
// draws (one lane).
__device__ __noinline__ void shuffle_wide(int32_t *a, uint32_t n, uint32_t run,
                                          uint32_t b, uint32_t k0, uint32_t k1)
{
    uint32_t w0 = 0, w1 = 0, w2 = 0, w3 = 0;
    uint32_t h = 4u, u = 0u;
    for (uint32_t j = n - 1u; j >= 1u; --j) {
        const uint32_t r = j + 1u;
        uint64_t m;
        for (;;) {
            if (h == 4u) {
                const u32x4 w = shuf_philox(u, run, b, 4u << 28, k0, k1);
                w0 = w.x;
                w1 = w.y;
                w2 = w.z;
                w3 = w.w;
                ++u;
                h = 0u;
            }
            const uint32_t x = h == 0u ? w0 : h == 1u ? w1 : h == 2u ? w2 : w3;
            ++h;
            m = (uint64_t)x * r;
            const uint32_t lo = (uint32_t)m;
            if (__builtin_expect(lo < r, 0) && lo < lemire_threshold32(r))
                continue;
            break;
        }
        const uint32_t k = (uint32_t)(m >> 32);
        const int32_t t = a[j];
        a[j] = a[k];
        a[k] = t;
    }
}

// Bucket labels of a chunk of elements: the wave's groups of 512 positions
// within the chunk, and its range.
struct ShufChunk {
    uint32_t g0, g1;  // the wave's group range (global group indices)
    uint32_t lo, hi;  // the chunk's element range
};

__device__ __forceinline__ ShufChunk shuf_chunk(uint32_t c, uint32_t M)
{
    const uint32_t wave = threadIdx.x >> 6;
    ShufChunk k;
    k.lo = c * SHUF_CHUNK;
    k.hi = min(M, k.lo + SHUF_CHUNK);
    const uint32_t first = k.lo / 512u, G = (k.hi - k.lo + 511u) / 512u;
    k.g0 = first + wave * G / SHUF_W;
    k.g1 = first + (wave + 1u) * G / SHUF_W;
    return k;
}

// Run and chunk of a count or scatter block: block g * 8 * chunks + 8 c + j
// is chunk c of run 8 g + j of the launch's rn runs, so the chunks of a run
// go to one XCD (workgroups are dealt to the 8 XCDs in turn) in chunk order.
// Both kernels write short pieces next to those of the neighbouring chunks
// (a count per bucket, a segment per bucket), and the lines they share fill
// up in that XCD's L2 instead of going out part-written.  False for the
// padding blocks of a last group of fewer than 8 runs.
__device__ __forceinline__ bool shuf_block(uint32_t chunks, uint32_t rn,
                                           uint32_t &rl, uint32_t &c)
{
    const uint32_t per_group = 8u * chunks;
    rl = blockIdx.x / per_group * 8u + blockIdx.x % 8u;
    c = blockIdx.x % per_group / 8u;
    return rl < rn;
}

__host__ __forceinline__ uint32_t shuf_blocks(uint32_t chunks, uint32_t rn)
{
    return (rn + 7u) / 8u * 8u * chunks;
}

// Count kernel: counts[(r * nb1 + b) * chunks + c] = elements of chunk c of
// run r with bucket label b.
__global__ __launch_bounds__(64 * SHUF_W) void shuffle_count_kernel(
    uint32_t k0, uint32_t k1, uint32_t first_run, uint32_t M, uint32_t lb1,
    uint32_t chunks, uint32_t r0, uint32_t rn, uint32_t *__restrict__ counts)
{
    extern __shared__ uint32_t cnt[];  // 2^lb1
    const uint32_t tid = threadIdx.x, lane = tid & 63u, nb1 = 1u << lb1;
    uint32_t rl, c;
    if (!shuf_block(chunks, rn, rl, c))
        return;
    const uint32_t r = r0 + rl, run = first_run + r;
    for (uint32_t i = tid; i < nb1; i += 64u * SHUF_W)
        cnt[i] = 0u;
    __syncthreads();
    const ShufChunk ch = shuf_chunk(c, M);
    for (uint32_t g = ch.g0; g < ch.g1; ++g) {
        const u32x4 key = lb1 ? shuf_philox((g << 6) | lane, run, 0u, 1u << 28, k0, k1)
                              : u32x4{0, 0, 0, 0};
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) {
            const uint32_t i = g * 512u + k * 64u + lane;
            if (i < ch.hi)
                atomicAdd(&cnt[lb1 ? half16(key, k) >> (16u - lb1) : 0u], 1u);
        }
    }
    __syncthreads();
    for (uint32_t b = tid; b < nb1; b += 64u * SHUF_W)
        counts[((uint64_t)r * nb1 + b) * chunks + c] = cnt[b];
}

// Scan kernel, one workgroup per run: counts become exclusive prefixes in
// (bucket major, chunk minor) order, starts[r * (nb1 + 1) + b] the first
// position of bucket b (starts[.. + nb1] = M).  Each wave reads whole
// buckets' chunk counts, 64 at a time (coalesced); bucket totals are
// scanned in LDS in between.
__global__ __launch_bounds__(256) void shuffle_scan_kernel(
    uint32_t M, uint32_t lb1, uint32_t chunks, uint32_t r0,
    uint32_t *__restrict__ counts, uint32_t *__restrict__ starts)
{
    extern __shared__ uint32_t tot[];  // 2^lb1 bucket totals, then bases
    __shared__ uint32_t wsum[4];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t r = r0 + blockIdx.x, nb1 = 1u << lb1;
    uint32_t *q = counts + (uint64_t)r * nb1 * chunks;
    uint32_t *st = starts + (uint64_t)r * (nb1 + 1u);
    for (uint32_t b = wave; b < nb1; b += 4u) {
        uint32_t acc = 0;
        for (uint32_t c = lane; c < chunks; c += 64u)
            acc += q[(uint64_t)b * chunks + c];
        acc = wave_scan_add(acc);
        if (lane == 63u)
            tot[b] = acc;
    }
    __syncthreads();
    {
        const uint32_t per = (nb1 + 255u) / 256u;
        const uint32_t a = min(tid * per, nb1), e = min(a + per, nb1);
        uint32_t sum = 0;
        for (uint32_t b = a; b < e; ++b)
            sum += tot[b];
        const uint32_t inc = wave_scan_add(sum);
        if (lane == 63u)
            wsum[wave] = inc;
        __syncthreads();
        uint32_t acc = inc - sum;
        for (uint32_t w = 0; w < wave; ++w)
            acc += wsum[w];
        for (uint32_t b = a; b < e; ++b) {
            const uint32_t t = tot[b];
            tot[b] = acc;
            st[b] = acc;
            acc += t;
        }
        if (tid == 0u)
            st[nb1] = M;
    }
    __syncthreads();
    for (uint32_t b = wave; b < nb1; b += 4u) {
        uint32_t carry = tot[b];
        for (uint32_t c0 = 0; c0 < chunks; c0 += 64u) {
            const uint32_t c = c0 + lane;
            const uint32_t v = c < chunks ? q[(uint64_t)b * chunks + c] : 0u;
            const uint32_t inc = wave_scan_add(v);
            if (c < chunks)
                q[(uint64_t)b * chunks + c] = carry + inc - v;
            carry += read_lane(inc, 63u);
        }
    }
}

// Scatter kernel: the elements of chunk c of run r, sorted by bucket label
// in LDS (stable), then written bucket by bucket with consecutive threads on
// consecutive addresses (whole cache lines, instead of one scattered 4-byte
// store per element); blocks laid out by shuf_block.
__global__ __launch_bounds__(64 * SHUF_W) void shuffle_scatter_kernel(
    uint32_t k0, uint32_t k1, uint32_t first_run, uint32_t M, uint32_t lb1,
    uint32_t chunks, uint32_t r0, uint32_t rn, const uint32_t *__restrict__ counts,
    int32_t *__restrict__ perm, int64_t stride)
{
    __shared__ unsigned long long masks[SHUF_W * MATCH_WORDS / 2u];
    __shared__ uint32_t sorted[SHUF_CHUNK];   // label << 16 | place in the chunk
    __shared__ uint32_t wsum[SHUF_W];
    extern __shared__ uint32_t dyn[];  // [SHUF_W][nb1] bases, [nb1] moves
    constexpr uint32_t GPW = SHUF_CHUNK / (512u * SHUF_W);
    const uint32_t T = 64u * SHUF_W, tid = threadIdx.x, lane = tid & 63u,
                   wave = tid >> 6;
    const uint32_t nb1 = 1u << lb1;
    uint32_t rl, c;
    if (!shuf_block(chunks, rn, rl, c))
        return;
    const uint32_t r = r0 + rl, run = first_run + r;
    uint32_t *base = dyn, *move = dyn + SHUF_W * nb1;
    uint32_t *my = base + wave * nb1;
    for (uint32_t i = tid; i < SHUF_W * nb1; i += T)
        base[i] = 0u;
    for (uint32_t i = tid; i < SHUF_W * MATCH_WORDS / 2u; i += T)
        masks[i] = 0ull;
    __syncthreads();
    const ShufChunk ch = shuf_chunk(c, M);
    u32x4 keys[GPW];
#pragma unroll
    for (uint32_t gi = 0; gi < GPW; ++gi) {
        const uint32_t g = ch.g0 + gi;
        keys[gi] = shuf_philox((g << 6) | lane, run, 0u, 1u << 28, k0, k1);
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) {
            const uint32_t i = g * 512u + k * 64u + lane;
            if (g < ch.g1 && i < ch.hi)
                atomicAdd(&my[half16(keys[gi], k) >> (16u - lb1)], 1u);
        }
    }
    __syncthreads();
    // local bucket starts (exclusive over buckets of the chunk's totals),
    // per-wave local bases, and from there to the chunk's place in the bucket
    {
        const uint32_t per = (nb1 + T - 1u) / T;
        const uint32_t a = min(tid * per, nb1), e = min(a + per, nb1);
        uint32_t sum = 0;
        for (uint32_t b = a; b < e; ++b)
            for (uint32_t w = 0; w < (uint32_t)SHUF_W; ++w)
                sum += base[w * nb1 + b];
        const uint32_t inc = wave_scan_add(sum);
        if (lane == 63u)
            wsum[wave] = inc;
        __syncthreads();
        uint32_t acc = inc - sum;
        for (uint32_t w = 0; w < wave; ++w)
            acc += wsum[w];
        for (uint32_t b = a; b < e; ++b) {
            move[b] = counts[((uint64_t)r * nb1 + b) * chunks + c] - acc;
            for (uint32_t w = 0; w < (uint32_t)SHUF_W; ++w) {
                const uint32_t n = base[w * nb1 + b];
                base[w * nb1 + b] = acc;
                acc += n;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t gi = 0; gi < GPW; ++gi) {
        const uint32_t g = ch.g0 + gi;
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) {
            const uint32_t i = g * 512u + k * 64u + lane;
            const bool ok = g < ch.g1 && i < ch.hi;
            const uint32_t bkt = half16(keys[gi], k) >> (16u - lb1);
            const uint64_t peers = match_label_lds(bkt, lb1, ok, masks + wave * (MATCH_WORDS / 2u));
            if (ok) {
                const uint32_t rank = lanes_below(peers);
                const uint32_t at = my[bkt];
                sorted[at + rank] = bkt << 16 | (i - ch.lo);
                if (rank == 0u)
                    my[bkt] = at + (uint32_t)__popcll(peers);
            }
        }
    }
    __syncthreads();
    int32_t *row = perm + (int64_t)r * stride;
    const uint32_t n = ch.hi - ch.lo;
    for (uint32_t t = tid; t < n; t += T) {
        const uint32_t v = sorted[t];
        row[move[v >> 16] + t] = (int32_t)(ch.lo + (v & 0xFFFFu));
    }
}

// Words per wave of the sub-bucket counters (16-bit, in pairs) for groups of
// at most cap elements.
__host__ __device__ __forceinline__ uint32_t shuf_hist_words(uint32_t cap)
{
    uint32_t lb = 0;
    while ((SHUF_SUB << lb) < cap)
        ++lb;
    return ((1u << lb) + 1u) / 2u;
}

// One bucket a[0..n), n <= the launch's cap, shuffled by a workgroup of W
// waves: sub-bucket labels, stable grouping of the local indices 0..n-1 in
// ent[] (16-bit), Fisher-Yates of each sub-bucket (one thread each), then
// a[t] = old a[ent[t]] (all loads in flight together, all stores after a
// barrier), or a[t] = ent[t] when a is the identity (IDENT: the whole run
// is one bucket).  hist holds W * hw words, wsum W, masks W tables of
// match_label_lds; GPW bounds the groups of 512 positions a wave labels.
template <int W, int GPW, bool IDENT>
__device__ void shuffle_group_lds(uint32_t n, uint32_t b, uint32_t run,
                                  uint32_t k0, uint32_t k1, int32_t *a,
                                  uint16_t *ent, uint32_t *hist, uint32_t hw,
                                  uint32_t *wsum, unsigned long long *masks,
                                  uint32_t in_lds)
{
    const uint32_t T = 64u * W, tid = threadIdx.x, wave = tid >> 6,
                   lane = tid & 63u;
    uint32_t lb = 0;
    while ((SHUF_SUB << lb) < n)
        ++lb;
    const uint32_t nb = 1u << lb;
    const uint32_t G = (n + 511u) / 512u;
    const uint32_t g0 = wave * G / W, g1 = (wave + 1u) * G / W;
    uint32_t *my = hist + wave * hw;

    for (uint32_t i = tid; i < W * hw; i += T)
        hist[i] = 0u;
    for (uint32_t i = tid; i < (uint32_t)W << in_lds; i += T)
        masks[i] = 0ull;
    __syncthreads();

    // labels of this wave's positions (8 per Philox call, kept for the
    // grouping below), counted per wave
    u32x4 keys[GPW];
#pragma unroll
    for (uint32_t gi = 0; gi < (uint32_t)GPW; ++gi) {
        const uint32_t g = g0 + gi;
        keys[gi] = (lb && g < g1)
                       ? shuf_philox((g << 6) | lane, run, b, 2u << 28, k0, k1)
                       : u32x4{0, 0, 0, 0};
        if (g < g1) {
#pragma unroll
            for (uint32_t k = 0; k < 8u; ++k) {
                const uint32_t j = g * 512u + k * 64u + lane;
                if (j < n) {
                    const uint32_t s = lb ? half16(keys[gi], k) >> (16u - lb) : 0u;
                    atomicAdd(&my[s >> 1], 1u << ((s & 1u) * 16u));
                }
            }
        }
    }
    __syncthreads();

    // exclusive prefix over (sub-bucket major, wave minor); each thread owns
    // whole words (both 16-bit counters of a sub-bucket pair, all waves)
    {
        const uint32_t pairs = (nb + 1u) / 2u;
        const uint32_t per = (pairs + T - 1u) / T;
        const uint32_t p0 = min(tid * per, pairs), p1 = min(p0 + per, pairs);
        uint32_t tot = 0;
        for (uint32_t p = p0; p < p1; ++p)
            for (uint32_t w = 0; w < (uint32_t)W; ++w) {
                const uint32_t word = hist[w * hw + p];
                tot += (word & 0xFFFFu) + (word >> 16);
            }
        const uint32_t inc = wave_scan_add(tot);
        if (lane == 63u)
            wsum[wave] = inc;
        __syncthreads();
        uint32_t run_ = inc - tot;
        for (uint32_t w = 0; w < wave; ++w)
            run_ += wsum[w];
        for (uint32_t p = p0; p < p1; ++p) {
            // sub-bucket 2p (low halves) of every wave, then 2p + 1 (high)
            uint32_t lo_total = 0;
            for (uint32_t w = 0; w < (uint32_t)W; ++w)
                lo_total += hist[w * hw + p] & 0xFFFFu;
            uint32_t a0 = run_, a1 = run_ + lo_total;
            for (uint32_t w = 0; w < (uint32_t)W; ++w) {
                const uint32_t word = hist[w * hw + p];
                hist[w * hw + p] = a0 | (a1 << 16);
                a0 += word & 0xFFFFu;
                a1 += word >> 16;
            }
            run_ = a1;
        }
    }
    __syncthreads();

    // stable grouping of the local indices: positions in increasing order,
    // rank among the lanes of the same label, the label's first lane
    // advances the wave's base
#pragma unroll
    for (uint32_t gi = 0; gi < (uint32_t)GPW; ++gi) {
        const uint32_t g = g0 + gi;
        if (g < g1) {
#pragma unroll
            for (uint32_t k = 0; k < 8u; ++k) {
                const uint32_t j = g * 512u + k * 64u + lane;
                const bool ok = j < n;
                const uint32_t s = lb ? half16(keys[gi], k) >> (16u - lb) : 0u;
                const uint64_t peers = match_label_lds(s, lb, ok, masks + (wave << in_lds), in_lds);
                if (ok) {
                    const uint32_t rank = lanes_below(peers);
                    const uint32_t sh = (s & 1u) * 16u;
                    const uint32_t at = (my[s >> 1] >> sh) & 0xFFFFu;
                    ent[at + rank] = (uint16_t)j;
                    if (rank == 0u)
                        atomicAdd(&my[s >> 1], (uint32_t)__popcll(peers) << sh);
                }
            }
        }
    }
    __syncthreads();

    // Fisher-Yates per sub-bucket: after the grouping the last wave's base
    // of sub-bucket s is the end of s
    const uint32_t *last = hist + (W - 1) * hw;
    for (uint32_t s = tid; s < nb; s += T) {
        const uint32_t en = (last[s >> 1] >> ((s & 1u) * 16u)) & 0xFFFFu;
        const uint32_t st =
            s ? (last[(s - 1u) >> 1] >> (((s - 1u) & 1u) * 16u)) & 0xFFFFu : 0u;
        if (en - st >= 2u)
            shuffle_sub(ent + st, en - st, st, run, b, k0, k1);
    }
    __syncthreads();

    if (IDENT) {
        for (uint32_t t = tid; t < n; t += T)
            a[t] = (int32_t)ent[t];
        return;
    }
    // a[t] = old a[ent[t]]: every load issued before any store of the
    // workgroup (the empty asm makes each thread wait for its loads before
    // the barrier)
    constexpr uint32_t GATHER = IDENT ? 1u : SHUF_GROUP_CAP / (64u * W);
    int32_t v[GATHER];
#pragma unroll
    for (uint32_t i = 0; i < GATHER; ++i) {
        const uint32_t t = tid + i * T;
        v[i] = t < n ? a[ent[t]] : 0;
    }
#pragma unroll
    for (uint32_t i = 0; i < GATHER; ++i)
        asm volatile("" ::"v"(v[i]));
    __syncthreads();
#pragma unroll
    for (uint32_t i = 0; i < GATHER; ++i) {
        const uint32_t t = tid + i * T;
        if (t < n)
            a[t] = v[i];
    }
}

// Group kernel: bucket b = blockIdx.x of run r0 + blockIdx.y, in place in
// the output row; cap bounds the buckets' sizes handled in LDS (the run's
// size when IDENT: one bucket, the identity before the shuffle).  Dynamic
// LDS: shuf_group_lds_bytes(W, cap).
template <int W, bool IDENT>
__global__ __launch_bounds__(64 * W) void shuffle_group_kernel(
    uint32_t k0, uint32_t k1, uint32_t first_run, uint32_t lb1, uint32_t r0,
    uint32_t cap, uint32_t in_lds, const uint32_t *__restrict__ starts,
    int32_t *__restrict__ perm, int64_t stride)
{
    extern __shared__ uint32_t gdyn[];
    constexpr uint32_t CAP =
        IDENT ? (W == 2 ? SHUF_SMALL_CAP : SHUF_WHOLE) : SHUF_GROUP_CAP;
    constexpr int GPW = (int)(CAP / (512u * W));
    const uint32_t hw = shuf_hist_words(cap);
    unsigned long long *masks = (unsigned long long *)gdyn;
    uint32_t *hist = gdyn + (2u * W << in_lds), *wsum = hist + W * hw;
    uint16_t *ent = (uint16_t *)(wsum + W);
    const uint32_t b = blockIdx.x, r = r0 + blockIdx.y;
    const uint32_t run = first_run + r;
    uint32_t o = 0, n = cap;
    if (!IDENT) {
        const uint32_t *st = starts + (uint64_t)r * ((1u << lb1) + 1u);
        o = st[b];
        n = st[b + 1u] - o;
    }
    int32_t *a = perm + (int64_t)r * stride + o;
    if (n <= 1u) {
        if (IDENT && n == 1u && threadIdx.x == 0u)
            a[0] = 0;
        return;
    }
    if (!IDENT && n > SHUF_GROUP_CAP) {
        if (threadIdx.x == 0u)
            shuffle_wide(a, n, run, b, k0, k1);
        return;
    }
    shuffle_group_lds<W, GPW, IDENT>(n, b, run, k0, k1, a, ent, hist, hw, wsum, masks,
                                     in_lds);
}

// (in_lds < 0: without the tables of match_label_lds)
static size_t shuf_group_lds_bytes(uint32_t W, uint32_t cap, int in_lds)
{
    const uint32_t table = in_lds < 0 ? 0u : 2u << in_lds;
    return (size_t)(W * (table + shuf_hist_words(cap)) + W) * 4u +
           (((size_t)cap * 2u + 3u) & ~(size_t)3u);
}

// Label bits matched through LDS in a workgroup of eight waves for a whole run
// of `cap` edges: fewer than MATCH_BITS, but at least 5, where a CU then holds
// as many workgroups as it would without the tables, and there are runs for
// them (40 of 21840 edges: 26.3 us with 7, 29.2 with 5).  4000 runs, microseconds
// with 7, 6 and 5 bits (and as the kernel was with ballots alone): 15312 edges
// 183, 173, 172 (184); 16380 196, 194, 186 (191); 20500 252, 234, 238 (262);
// 21424 264, 275, 247 (272); 32768 543, 403, 415 (469).  With 4 bits the lanes
// that wait for each other cost more than the workgroup is worth: 22500 edges
// 272 with 7, 303.
static uint32_t shuf_match_bits(uint32_t cap, uint32_t num_runs)
{
    constexpr uint32_t LDS = 160u << 10, WAVES = 2048u / 512u, CUS = 256u;
    auto resident = [&](int in_lds) {
        return std::min<size_t>(LDS / shuf_group_lds_bytes(8, cap, in_lds), WAVES);
    };
    if (num_runs <= CUS * resident(MATCH_BITS))
        return MATCH_BITS;
    for (int bits = MATCH_BITS; bits >= 5; --bits)
        if (resident(bits) == resident(-1))
            return (uint32_t)bits;
    return MATCH_BITS;
}

// ---------------------------------------------------------------------------
// Bit-exact device permutations: numpy's legacy RandomState(seed).permutation
// (the permutations the reference draws, percolate/hpc.py:195,206).
// MT19937 (Matsumoto & Nishimura, 1998) seeded with init_genrand(seed), as
// RandomState does for an integer seed; permutation(n) shuffles arange(n)
// from the end: for i = n-1 .. 1, j is the first 32-bit draw whose low bits
// under the smallest all-ones mask >= i are <= i, then a[i] and a[j] swap.
// One run per wavefront: the 624-word twist is computed by all lanes in four
// phases that respect the recurrence's order, the draws are consumed on
// uniform (scalar) control flow and lane 0 performs the swaps, in LDS
// (16-bit entries, n <= 65536) or in the output row.
// ---------------------------------------------------------------------------
#define MT_N 624
#define MT_SHIFT 397
#define MT_LDS_MAX 65536u

__device__ __forceinline__ uint32_t mt_next_word(uint32_t cur, uint32_t nxt,
                                                 uint32_t far)
{
    const uint32_t y = (cur & 0x80000000u) | (nxt & 0x7fffffffu);
    return far ^ (y >> 1) ^ ((y & 1u) ? 0x9908b0dfu : 0u);
}

// new mt[k] for k in [lo, hi), reading mt[k + 397] (k < 227) or the already
// renewed mt[k - 227] (k >= 227)
__device__ __forceinline__ void mt_twist_range(uint32_t *mt, uint32_t lo,
                                               uint32_t hi)
{
    for (uint32_t k0 = lo; k0 < hi; k0 += 64u) {
        const uint32_t k = k0 + threadIdx.x;
        uint32_t v = 0;
        if (k < hi)
            v = mt_next_word(mt[k], mt[k + 1u == MT_N ? 0u : k + 1u],
                             mt[k < MT_N - MT_SHIFT ? k + MT_SHIFT : k - (MT_N - MT_SHIFT)]);
        if (k < hi)
            mt[k] = v;
    }
}

__device__ __forceinline__ void mt_twist(uint32_t *mt)
{
    mt_twist_range(mt, 0u, MT_N - MT_SHIFT);        // 0..226: old words
    mt_twist_range(mt, MT_N - MT_SHIFT, 2u * (MT_N - MT_SHIFT)); // 227..453
    mt_twist_range(mt, 2u * (MT_N - MT_SHIFT), MT_N - 1u);      // 454..622
    mt_twist_range(mt, MT_N - 1u, MT_N);            // 623: renewed mt[0], mt[396]
}

__device__ __forceinline__ uint32_t mt_temper(uint32_t y)
{
    y ^= y >> 11;
    y ^= (y << 7) & 0x9d2c5680u;
    y ^= (y << 15) & 0xefc60000u;
    y ^= y >> 18;
    return y;
}

template <bool LDS_ARRAY>
__global__ __launch_bounds__(64) void permute_randomstate_kernel(
    const uint32_t *__restrict__ seeds, uint32_t n, int32_t *__restrict__ perm,
    int64_t stride)
{
    __shared__ uint32_t mt[MT_N];
    extern __shared__ uint16_t arr16[];
    const uint32_t lane = threadIdx.x;
    int32_t *out = perm + (int64_t)blockIdx.x * stride;
    if (lane == 0) {
        uint32_t x = seeds[blockIdx.x];
        mt[0] = x;
        for (uint32_t i = 1; i < MT_N; ++i) {
            x = 1812433253u * (x ^ (x >> 30)) + i;
            mt[i] = x;
        }
    }
    for (uint32_t i = lane; i < n; i += 64u) {
        if (LDS_ARRAY)
            arr16[i] = (uint16_t)i;
        else
            out[i] = (int32_t)i;
    }
    __syncthreads();

    // The draws do not depend on the array: the wave tempers the next 64
    // words of the state at once (lane k holds word base + k) and each draw
    // is a lane read, so the only LDS round trip per step is the swap's.
    uint32_t pos = MT_N, base = MT_N;
    uint32_t buf = 0;
    uint32_t i = n ? n - 1u : 0u;
    while (i >= 1u) {
        uint32_t mask = i;
        mask |= mask >> 1;
        mask |= mask >> 2;
        mask |= mask >> 4;
        mask |= mask >> 8;
        mask |= mask >> 16;
        uint32_t v;
        do {
            if (pos == MT_N) {
                __syncthreads();
                mt_twist(mt);
                __syncthreads();
                pos = 0;
                base = MT_N;
            }
            if (pos - base >= 64u) {
                // refill (base = MT_N after a twist makes pos - base wrap)
                base = pos;
                buf = base + lane < MT_N ? mt_temper(mt[base + lane]) : 0u;
            }
            v = read_lane(buf, pos - base) & mask;
            ++pos;
        } while (v > i);
        if (lane == 0) {
            if (LDS_ARRAY) {
                const uint16_t a = arr16[i], b = arr16[v];
                arr16[i] = b;
                arr16[v] = a;
            } else {
                const int32_t a = out[i], b = out[v];
                out[i] = b;
                out[v] = a;
            }
        }
        --i;
    }
    if (LDS_ARRAY) {
        __syncthreads();
        for (uint32_t k = lane; k < n; k += 64u)
            out[k] = (int32_t)arr16[k];
    }
}

// The same permutation in two parallel phases (runs of at most
// RS_APPLY_MAX edges).  The shuffle's swap targets depend on the MT19937
// stream alone, not on the array: phase one draws them (one wavefront per
// run) and stores the target k_i of step i in the output row; phase two
// applies all swaps at once.  Steps run i = n-1 .. 1 and step i writes only
// positions i and k_i <= i, so no later step writes position i again and
// the result at position i >= 1 is the value position k_i holds just before
// step i.  The writers of a position p before step i are the steps s > i
// with k_s = p, the last of them being the smallest; the value such a step
// s brings to p is the one position s holds just before step s.  With
//   F(p) = the smallest step s > p with k_s = p (none possible),
//   V(p) = the value position p holds just before step p
//        = V(F(p)), or p itself when F(p) does not exist,
// V is the root of p's chain p -> F(p) -> F(F(p)) ... (F only increases),
// the result at i >= 1 is V(s) for the smallest step s > i with k_s = k_i,
// or k_i itself without one, and the result at 0 is V(0).
#define RS_APPLY_MAX 32768u

// The first words of MT19937 for a seed (init_genrand), by one wavefront: the
// chain of 624 dependent steps runs on the scalar unit, a lane of a register
// takes each word, and 64 words are stored at a time.
__device__ __forceinline__ void mt_init(uint32_t seed, uint32_t *mt)
{
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t x = uniform(seed);
#pragma nounroll
    for (uint32_t b = 0; b < MT_N; b += 64u) {
        uint32_t v = 0;
#pragma unroll
        for (uint32_t l = 0; l < 64u; ++l) {
            asm("v_writelane_b32 %0, %1, %2" : "+v"(v) : "s"(x), "i"(l));
            x = 1812433253u * (x ^ (x >> 30)) + (b + l + 1u);
        }
        if (b + lane < MT_N)
            mt[b + lane] = v;
    }
}

// Phase one.  The wave tempers 64 state words at a time (lane l holds word
// base + l) and settles the whole block at once: for steps i, i-1, ... under
// one mask m (the smallest all-ones mask >= i), the word of lane l serves
// step i - (accepted words below l), so x = word & m is accepted for sure
// when x <= i - 63, rejected for sure when x > i, and the lanes in between are
// narrowed down together (a lane at a time, 40 runs of 480 edges took 36 us,
// not 17, and 4000 of 32512 0.51 ms, not 0.42).  The mask holds for c = i - m/2 more steps; when the
// block accepts c words or more, the lanes after the c-th accepted one are
// settled again under the next mask.
// mt_settle takes the words of one twist so; it returns the step reached.
__device__ __forceinline__ uint32_t mt_settle(const uint32_t *mt, uint32_t i, int32_t *out)
{
    const uint32_t lane = threadIdx.x & 63u;
    for (uint32_t pos = 0; pos < MT_N && i >= 1u;) {
        const uint32_t nw = min(64u, MT_N - pos);
        const uint32_t w = lane < nw ? mt_temper(mt[pos + lane]) : 0u;
        uint32_t l0 = 0;
        do {
            const uint32_t m = 0xFFFFFFFFu >> __builtin_clz(i);
            const uint32_t c = i - (m >> 1);
            const uint32_t x = w & m;
            const bool valid = lane >= l0 && lane < nw;
            // accepted for sure and perhaps: with as many accepted below as
            // there may be, and with as few.  Each turn settles at least the
            // first lane in doubt, most turns nearly all of them.
            uint64_t acc = ballot(valid && x + 63u <= i);
            uint64_t may = ballot(valid && x <= i);
            while (acc != may) {
                const uint32_t most = lanes_below(may), least = lanes_below(acc);
                acc = ballot(valid && x + most <= i);
                may = ballot(valid && x + least <= i);
            }
            const uint32_t below = lanes_below(acc);
            const bool mine = (acc >> lane) & 1ull;
            const uint32_t cnt = (uint32_t)__popcll(acc);
            uint32_t used;
            if (cnt >= c) {
                // the c-th accepted lane takes the mask's last step
                const uint32_t last = (uint32_t)__builtin_ctzll(ballot(mine && below == c - 1u));
                if (mine && below < c)
                    out[i - below] = (int32_t)x;
                used = c;
                l0 = last + 1u;
            } else {
                if (mine)
                    out[i - below] = (int32_t)x;
                used = cnt;
                l0 = nw;
            }
            i -= used;
        } while (l0 < nw && i >= 1u);
        pos += nw;
    }
    return i;
}

__global__ __launch_bounds__(64) void randomstate_targets_kernel(
    const uint32_t *__restrict__ seeds, uint32_t n, int32_t *__restrict__ perm,
    int64_t stride)
{
    __shared__ uint32_t mt[MT_N];
    int32_t *out = perm + (int64_t)blockIdx.x * stride;
    mt_init(seeds[blockIdx.x], mt);
    if (threadIdx.x == 0u && n)
        out[0] = 0;
    uint32_t i = n ? n - 1u : 0u;
    while (i >= 1u) {
        __syncthreads();
        mt_twist(mt);
        __syncthreads();
        i = mt_settle(mt, i, out);
    }
}

// Phase one by a workgroup of 640 threads, thread t with state word t: a
// twist is three steps of all threads (two barriers), and the 624 words are
// settled together where the mask holds for all of them.  The word at place t
// serves step i - (accepted words below t), of which there are at most t: it
// is accepted for sure when x + t <= i, rejected for sure when x > i, and the
// few in between (about 624^2 / 2 of every m + 1 words' worth) are decided in
// order by the first wavefront.  Words around a change of mask, and the last
// RST_SMALL steps, go through the blocks of 64 above on that wavefront.
#define RST_T 640u
#define RST_SMALL 8192u

__global__ __launch_bounds__(RST_T) void randomstate_targets_wide_kernel(
    const uint32_t *__restrict__ seeds, uint32_t n, int32_t *__restrict__ perm,
    int64_t stride)
{
    constexpr uint32_t WAVES = RST_T / 64u, OUT = MT_N - MT_SHIFT;
    __shared__ uint32_t mt[2][MT_N];
    __shared__ uint32_t xs[RST_T];
    __shared__ uint64_t accepted[WAVES], open[WAVES];
    __shared__ uint32_t before[WAVES + 1u];
    const uint32_t t = threadIdx.x, wave = uniform(t >> 6);
    int32_t *out = perm + (int64_t)blockIdx.x * stride;
    if (wave == 0u)
        mt_init(seeds[blockIdx.x], mt[0]);
    if (t == 0u && n)
        out[0] = 0;
    __syncthreads();
    uint32_t i = n ? n - 1u : 0u;
    for (uint32_t g = 0; i >= 1u; ++g) {
        const uint32_t *old = mt[g & 1u];
        uint32_t *now = mt[(g + 1u) & 1u];
        uint32_t a = 0, b = 0, y = 0;
        if (t < MT_N) {
            a = old[t];
            b = old[t + 1u < MT_N ? t + 1u : 0u];
        }
        if (t < OUT)
            now[t] = y = mt_next_word(a, b, old[t + MT_SHIFT]);
        __syncthreads();
        if (t >= OUT && t < 2u * OUT)
            now[t] = y = mt_next_word(a, b, now[t - OUT]);
        __syncthreads();
        if (t >= 2u * OUT && t < MT_N)
            now[t] = y = mt_next_word(a, t + 1u < MT_N ? b : now[0], now[t - OUT]);
        const uint32_t m = 0xFFFFFFFFu >> __builtin_clz(i);
        if (i >= RST_SMALL && i - (m >> 1) > MT_N) {
            const uint32_t x = mt_temper(y) & m;
            const bool in = t < MT_N;
            const uint64_t acc = ballot(in && x + t <= i);
            const uint64_t amb = ballot(in && x <= i && x + t > i);
            xs[t] = x;
            if ((t & 63u) == 0u) {
                accepted[wave] = acc;
                open[wave] = amb;
            }
            __syncthreads();
            if (wave == 0u) {
                const uint32_t l = min(t, WAVES - 1u);
                const uint64_t all = accepted[l], some = open[l];
                uint32_t base = 0, at = 0;
                uint64_t fin = 0;
#pragma unroll
                for (uint32_t w = 0; w < WAVES; ++w) {
                    uint64_t ok = read_lane(all, w), left = read_lane(some, w);
                    while (left) {
                        const uint32_t z = (uint32_t)__builtin_ctzll(left);
                        const uint32_t below = (uint32_t)__popcll(ok & ((1ull << z) - 1ull));
                        if (uniform(xs[w * 64u + z]) + base + below <= i)
                            ok |= 1ull << z;
                        left &= left - 1ull;
                    }
                    if (t == w) {
                        fin = ok;
                        at = base;
                    }
                    base += (uint32_t)__popcll(ok);
                }
                if (t < WAVES) {
                    accepted[t] = fin;
                    before[t] = at;
                }
                if (t == 0u)
                    before[WAVES] = base;
            }
            __syncthreads();
            const uint64_t fin = accepted[wave];
            if ((fin >> (t & 63u)) & 1ull)
                out[i - before[wave] - lanes_below(fin)] = (int32_t)x;
            i -= uniform(before[WAVES]);
        } else {
            __syncthreads();
            if (wave == 0u) {
                const uint32_t r = mt_settle(now, i, out);
                if (t == 0u)
                    before[WAVES] = r;
            }
            __syncthreads();
            i = uniform(before[WAVES]);
        }
    }
}

// Smallest of the list entries ent[b..e) above thr, or 0xFFFF (entries are
// steps, 1 <= s < n <= 32768), and whether an entry below thr exists; four
// entries are read per round.
__device__ __forceinline__ uint32_t rs_list_scan(const uint16_t *ent, uint32_t b,
                                                 uint32_t e, uint32_t thr, bool &below)
{
    uint32_t best = 0xFFFFu;
    bool lo = false;
    for (uint32_t a = b; a < e; a += 4u) {
        uint32_t x[4];
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u)
            x[u] = ent[min(a + u, e - 1u)];
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u) {
            best = x[u] > thr ? min(best, x[u]) : best;
            lo |= x[u] < thr;
        }
    }
    below = lo;
    return best;
}

// A copy of x the compiler cannot relate to x: predicates computed from it in
// one phase are not kept alive (as 32 lane masks) for a later phase.
__device__ __forceinline__ uint32_t opaque(uint32_t x)
{
    asm volatile("" : "+s"(x));
    return x;
}
__device__ __forceinline__ uint32_t opaque_v(uint32_t x)
{
    asm volatile("" : "+v"(x));
    return x;
}

// Phase two, one workgroup of T threads per run of n <= T * PER edges, in place over the targets.  LDS holds 16-bit list cursors of the
// positions in pairs and the lists of steps per target position (a counting
// sort: counts, exclusive scan, placement; unordered within a list); every
// thread owns indices j = tid + q * T (q < PER) and scans the list of k_j
// once, for the smallest step above j and for whether j is the list's
// smallest step (which then knows F(k_j)).  The list area is then reused for
// V, which pointer jumping (V(p) <- V(V(p)) until nothing changes, over
// position pairs) takes to the chain roots.  The loads of independent items
// are issued together before any is waited for.  Dynamic LDS:
// rs_apply_lds_bytes(n).
template <uint32_t T, uint32_t PER>
__global__ __launch_bounds__(T) void randomstate_apply_kernel(
    uint32_t n, int32_t *__restrict__ perm, int64_t stride)
{
    constexpr uint32_t PAIRS = PER / 2u, WAVES = T / 64u, LOOKUP = 0x8000u;
    constexpr uint32_t GROUP = PER < 4u ? PER : 4u;
    extern __shared__ uint32_t rsd[];
    const uint32_t words = (n + 2u) / 2u;   // 16-bit cursors of positions 0..n
    uint32_t *cur = rsd;
    uint16_t *ent = (uint16_t *)(rsd + words);
    uint32_t *V2 = rsd + words;             // V of positions 2w, 2w + 1
    const uint16_t *V = ent;
    __shared__ uint32_t wsum[WAVES];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    int32_t *row = perm + (int64_t)blockIdx.x * stride;
    if (n == 0u)
        return;
    const uint32_t npairs = (n + 1u) / 2u;
    uint32_t k[PER];
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q) {
        const uint32_t j = tid + q * T;
        const uint32_t v = (uint32_t)row[min(j, n - 1u)];
        k[q] = (j >= 1u && j < n) ? v : 0u;
    }
    for (uint32_t w = tid; w < words; w += T)
        cur[w] = 0u;
    __syncthreads();
    // steps per target position
    {
        const uint32_t nn = opaque(n), t0 = opaque_v(tid);
#pragma unroll
        for (uint32_t q = 0; q < PER; ++q) {
            const uint32_t j = t0 + q * T;
            if (j >= 1u && j < nn)
                atomicAdd(&cur[k[q] >> 1], 1u << ((k[q] & 1u) * 16u));
        }
    }
    __syncthreads();
    // exclusive prefix: cur[p] = first slot of position p's list.  Wave w
    // scans words [w * chunk, (w + 1) * chunk), 64 consecutive words per
    // round, after one pass for the wave totals.
    {
        const uint32_t chunk = ((words + WAVES - 1u) / WAVES + 63u) & ~63u;
        const uint32_t w0 = min(wave * chunk, words), w1 = min(w0 + chunk, words);
        uint32_t tot = 0;
        for (uint32_t w = w0 + lane; w < w1; w += 64u) {
            const uint32_t x = cur[w];
            tot += (x & 0xFFFFu) + (x >> 16);
        }
        tot = read_lane(wave_scan_add(tot), 63u);
        if (lane == 0u)
            wsum[wave] = tot;
        __syncthreads();
        uint32_t carry = 0;
        for (uint32_t w = 0; w < wave; ++w)
            carry += wsum[w];
        for (uint32_t b = w0; b < w1; b += 64u) {
            const uint32_t w = b + lane;
            const uint32_t x = w < w1 ? cur[w] : 0u;
            const uint32_t pair = (x & 0xFFFFu) + (x >> 16);
            const uint32_t inc = wave_scan_add(pair);
            const uint32_t a0 = carry + inc - pair, a1 = a0 + (x & 0xFFFFu);
            if (w < w1)
                cur[w] = a0 | (a1 << 16);
            carry += read_lane(inc, 63u);
        }
    }
    __syncthreads();
    // place the steps; afterwards cursor p is the end of p's list, which is
    // where p + 1's list starts
    const uint32_t np = opaque(n), tp = opaque_v(tid);
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q) {
        const uint32_t j = tp + q * T;
        if (j >= 1u && j < np) {
            const uint32_t sh = (k[q] & 1u) * 16u;
            const uint32_t at = (atomicAdd(&cur[k[q] >> 1], 1u << sh) >> sh) & 0xFFFFu;
            ent[at] = (uint16_t)j;
        }
    }
    __syncthreads();
    // Each step j scans the list of its target p = k_j once: the smallest
    // step above j there (its successor), and whether j is the list's
    // smallest step, in which case j knows F(p): j itself when j > p, else
    // (j = p) its successor.  Per index, packed: low half the result, or
    // LOOKUP | s for "V(s)"; bit 31 set for a list's smallest step, with
    // F(p) in bits 16..30 (all values are below 2^15).  The list bounds of a
    // group of indices are read before the lists.
    auto half = [&](uint32_t x, uint32_t p) { return (x >> ((p & 1u) * 16u)) & 0xFFFFu; };
    uint32_t rf[PER];
    const uint32_t nr = opaque(n), tr = opaque_v(tid);
#pragma unroll
    for (uint32_t g = 0; g < PER; g += GROUP) {
        uint32_t se[GROUP], sb[GROUP];
#pragma unroll
        for (uint32_t u = 0; u < GROUP; ++u) {
            const uint32_t p = k[g + u];
            se[u] = cur[p >> 1];
            sb[u] = cur[p ? (p - 1u) >> 1 : 0u];     // unused for p = 0
        }
#pragma unroll
        for (uint32_t u = 0; u < GROUP; ++u) {
            const uint32_t q = g + u, j = tr + q * T;
            uint32_t r = LOOKUP, w = 0u;
            if (j < nr && j) {
                const uint32_t p = k[q];
                const uint32_t b = p ? half(sb[u], p - 1u) : 0u, e = half(se[u], p);
                bool below;
                const uint32_t s = rs_list_scan(ent, b, e, j, below);
                r = s == 0xFFFFu ? p : (LOOKUP | s);
                if (!below)
                    w = 0x80000000u | ((j > p ? j : (s == 0xFFFFu ? p : s)) << 16);
            }
            rf[q] = r | w;
        }
    }
    __syncthreads();
    // the results move to the cursor area; V, in the list area, starts as
    // every position itself (the positions no step targets keep that), then
    // each list's smallest step writes F of its target
    uint16_t *res = (uint16_t *)cur;
    {
        uint16_t *Vw = ent;
        const uint32_t nv = opaque(n), tv = opaque_v(tid);
#pragma unroll
        for (uint32_t q = 0; q < PER; ++q) {
            const uint32_t j = tv + q * T;
            if (j < nv) {
                res[j] = (uint16_t)rf[q];
                Vw[j] = (uint16_t)j;
            }
        }
        __syncthreads();
#pragma unroll
        for (uint32_t q = 0; q < PER; ++q)
            if (rf[q] >> 31)
                Vw[k[q]] = (uint16_t)((rf[q] >> 16) & 0x7FFFu);
    }
    __syncthreads();
    // pointer jumping over the pairs; a concurrent update only moves a
    // pointer further up its own chain, and a round without a change leaves
    // every pointer at a root.  An odd n's last pair has a padding half,
    // kept as it is.
    for (;;) {
        uint32_t v[PAIRS], y0[PAIRS], y1[PAIRS];
        const uint32_t tj = opaque_v(tid);
#pragma unroll
        for (uint32_t h = 0; h < PAIRS; ++h)
            v[h] = V2[min(tj + h * T, npairs - 1u)];
#pragma unroll
        for (uint32_t h = 0; h < PAIRS; ++h) {
            y0[h] = V[v[h] & 0xFFFFu];
            y1[h] = V[min(v[h] >> 16, n - 1u)];
        }
        bool changed = false;
#pragma unroll
        for (uint32_t h = 0; h < PAIRS; ++h) {
            const uint32_t w = tj + h * T;
            const uint32_t hi = 2u * w + 1u < n ? y1[h] : v[h] >> 16;
            const uint32_t nv = y0[h] | (hi << 16);
            const bool c = w < npairs && nv != v[h];
            if (c)
                V2[w] = nv;
            changed |= c;
        }
        if (!__syncthreads_or(changed))
            break;
    }
    const uint32_t tf = opaque_v(tid);
#pragma unroll
    for (uint32_t g = 0; g < PER; g += GROUP) {
        uint32_t r[GROUP], val[GROUP];
#pragma unroll
        for (uint32_t u = 0; u < GROUP; ++u)
            r[u] = res[min(tf + (g + u) * T, n - 1u)];
#pragma unroll
        for (uint32_t u = 0; u < GROUP; ++u)
            val[u] = (r[u] & LOOKUP) ? (uint32_t)V[min(r[u] & ~LOOKUP, n - 1u)] : r[u];
#pragma unroll
        for (uint32_t u = 0; u < GROUP; ++u) {
            const uint32_t j = tf + (g + u) * T;
            if (j < n)
                row[j] = (int32_t)val[u];
        }
    }
}

// The second phase for runs of more than RS_APPLY_MAX edges, which one
// workgroup's LDS does not hold: positions are cut into buckets of at most
// RSB_CAP positions and about as many steps targeting them, and one workgroup
// per run takes the buckets from the top position down.  The steps of a run
// are first grouped by the bucket of their target in the workspace; a bucket
// is then the whole of phase two for its positions: the lists of its
// positions (a counting sort in LDS), each step's successor and each
// position's F from the lists, and V.  F(p) > p is a position of the same
// bucket, resolved by pointer jumping in LDS, or of one done before, whose V
// is in the workspace; so is the position whose V is a step's result.  The
// result goes to the row, whose targets have all been read by then.
// Bound by the LDS and barrier latencies of a bucket (about 20 us of a
// workgroup each, 33 buckets at L = 256): 200 runs of L = 256 take 0.73 ms,
// where the swaps walked in sequence took 37 ms; 512 threads instead of 1024
// 0.87 ms.
//
// Buckets: the steps i >= x target a position below x with probability
// x / (i + 1), so x + x ln(n / x) targets below x are expected; a bucket
// spans RSB_WIDTH expected steps, or RSB_WIDTH positions near the top, where
// fewer steps than positions remain.  Its bounds are multiples of a cell of
// 2^shift positions (at most RSB_CELLS cells); the first cell holds up to
// 2560 steps (2^21 edges), so at most 7760 steps are expected, and more than
// RSB_CAP are 4.9 standard deviations off; the run is then walked in sequence.
#define RSB_T 1024u
#define RSB_CAP 8192u
#define RSB_WIDTH 5200u
#define RSB_CELLS 8192u
#define RSB_BUCKETS 1024u
#define RSB_MAX (1u << 21)
#define RSB_SHORT (1u << 19)   // up to so many edges an entry has 32 bits

struct RsbTable {
    uint32_t nb;
    uint32_t bounds[RSB_BUCKETS + 1u];
    uint16_t cell[RSB_CELLS];
};

__device__ __forceinline__ uint32_t rsb_bucket(double x, double n)
{
    // expected steps below x, then positions, past the point n / e where a
    // position expects one step
    const double e = n * 0.36787944117144233, at = min(x, e);
    const double g = at > 0.0 ? at + at * log(n / at) : 0.0;
    return (uint32_t)((g + max(x - e, 0.0)) / (double)RSB_WIDTH);
}

__global__ __launch_bounds__(256) void randomstate_table_kernel(uint32_t n, uint32_t shift,
                                                                RsbTable *__restrict__ t)
{
    const uint32_t cells = ((n - 1u) >> shift) + 1u;
    for (uint32_t c = blockIdx.x * 256u + threadIdx.x; c < cells; c += gridDim.x * 256u) {
        const uint32_t b = rsb_bucket((double)(c << shift), (double)n);
        const uint32_t before = c ? rsb_bucket((double)((c - 1u) << shift), (double)n) : 0u;
        t->cell[c] = (uint16_t)b;
        if (c == 0u)
            t->bounds[0] = 0u;
        for (uint32_t j = before + 1u; j <= b; ++j)
            t->bounds[j] = c << shift;
        if (c + 1u == cells) {
            t->nb = b + 1u;
            t->bounds[b + 1u] = n;
        }
    }
}

// Smallest of the list entries ent[b..e) above thr, or all ones, and whether
// an entry below thr exists.
__device__ __forceinline__ uint32_t rsb_list_scan(const uint32_t *ent, uint32_t b,
                                                  uint32_t e, uint32_t thr, bool &below)
{
    uint32_t best = 0xFFFFFFFFu;
    bool lo = false;
    for (uint32_t a = b; a < e; a += 2u) {
        const uint32_t x = ent[a], y = ent[min(a + 1u, e - 1u)];
        best = x > thr ? min(best, x) : best;
        best = y > thr ? min(best, y) : best;
        lo |= x < thr || y < thr;
    }
    below = lo;
    return best;
}

template <typename ENT>
__global__ __launch_bounds__(RSB_T) void randomstate_buckets_kernel(
    uint32_t n, uint32_t runs, uint32_t shift, const RsbTable *__restrict__ table,
    ENT *__restrict__ entries, uint32_t *values, int32_t *perm, int64_t stride)
{
    constexpr uint32_t T = RSB_T, PER = RSB_CAP / T, WAVES = T / 64u, DONE = 0x80000000u;
    constexpr uint32_t STEP_BITS = sizeof(ENT) == 4u ? 19u : 32u;
    __shared__ uint16_t cell[RSB_CELLS];
    __shared__ uint32_t bounds[RSB_BUCKETS + 1u], start[RSB_BUCKETS + 1u], next[RSB_BUCKETS];
    __shared__ uint32_t cur[RSB_CAP / 2u + 1u];   // 16-bit list cursors
    __shared__ uint32_t list[RSB_CAP];            // the lists, then V
    __shared__ uint32_t wsum[WAVES];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t nb = table->nb, cells = ((n - 1u) >> shift) + 1u;
    for (uint32_t c = tid; c < cells; c += T)
        cell[c] = table->cell[c];
    for (uint32_t b = tid; b <= nb; b += T)
        bounds[b] = table->bounds[b];
    ENT *ent = entries + (size_t)blockIdx.x * n;
    uint32_t *V = values + (size_t)blockIdx.x * n;
    for (uint32_t run = blockIdx.x; run < runs; run += gridDim.x) {
        int32_t *row = perm + (int64_t)run * stride;
        for (uint32_t b = tid; b < nb; b += T)
            next[b] = 0u;
        __syncthreads();
        // steps per bucket
        for (uint32_t i0 = 0; i0 < n; i0 += 8u * T) {
            uint32_t k[8];
#pragma unroll
            for (uint32_t u = 0; u < 8u; ++u)
                k[u] = (uint32_t)row[min(i0 + u * T + tid, n - 1u)];
#pragma unroll
            for (uint32_t u = 0; u < 8u; ++u) {
                const uint32_t i = i0 + u * T + tid;
                if (i >= 1u && i < n)
                    atomicAdd(&next[cell[k[u] >> shift]], 1u);
            }
        }
        __syncthreads();
        // their first entries; a thread owns two buckets
        static_assert(2u * T >= RSB_BUCKETS, "two buckets a thread");
        bool over = false;
        {
            const uint32_t c0 = 2u * tid < nb ? next[2u * tid] : 0u;
            const uint32_t c1 = 2u * tid + 1u < nb ? next[2u * tid + 1u] : 0u;
            over = c0 > RSB_CAP || c1 > RSB_CAP;
            const uint32_t inc = wave_scan_add(c0 + c1);
            if (lane == 63u)
                wsum[wave] = inc;
            __syncthreads();
            uint32_t a = inc - c0 - c1;
            for (uint32_t w = 0; w < wave; ++w)
                a += wsum[w];
            if (2u * tid < nb)
                start[2u * tid] = next[2u * tid] = a;
            if (2u * tid + 1u < nb)
                start[2u * tid + 1u] = next[2u * tid + 1u] = a + c0;
            if (tid == 0u)
                start[nb] = n - 1u;
        }
        if (__syncthreads_or(over)) {
            for (uint32_t j = tid; j < n; j += T)
                V[j] = j;
            __threadfence_block();
            __syncthreads();
            if (tid == 0u)
                for (uint32_t i = n - 1u; i >= 1u; --i) {
                    const uint32_t k = (uint32_t)row[i], a = V[i];
                    V[i] = V[k];
                    V[k] = a;
                }
            __threadfence_block();
            __syncthreads();
            for (uint32_t j = tid; j < n; j += T)
                row[j] = (int32_t)V[j];
            __syncthreads();
            continue;
        }
        // the steps grouped by bucket: step, and place of the target in it
        for (uint32_t i0 = 0; i0 < n; i0 += 8u * T) {
            uint32_t k[8];
#pragma unroll
            for (uint32_t u = 0; u < 8u; ++u)
                k[u] = (uint32_t)row[min(i0 + u * T + tid, n - 1u)];
#pragma unroll
            for (uint32_t u = 0; u < 8u; ++u) {
                const uint32_t i = i0 + u * T + tid;
                if (i >= 1u && i < n) {
                    const uint32_t b = cell[k[u] >> shift];
                    ent[atomicAdd(&next[b], 1u)] = (ENT)i | ((ENT)(k[u] - bounds[b]) << STEP_BITS);
                }
            }
        }
        __threadfence_block();
        __syncthreads();
        for (uint32_t b = nb; b-- > 0u;) {
            const uint32_t lo = bounds[b], hi = bounds[b + 1u], W = hi - lo;
            const uint32_t s0 = start[b], E = start[b + 1u] - s0;
            if (W == 0u)
                continue;
            const uint32_t words = (W + 1u) / 2u;
            uint32_t step[PER], pos[PER], succ[PER], first[PER];
#pragma unroll
            for (uint32_t q = 0; q < PER; ++q)
                if (q * T < E) {
                    const ENT e = ent[s0 + min(q * T + tid, E - 1u)];
                    step[q] = (uint32_t)(e & (ENT)((1ull << STEP_BITS) - 1u));
                    pos[q] = (uint32_t)((uint64_t)e >> STEP_BITS);
                }
            for (uint32_t w = tid; w < words; w += T)
                cur[w] = 0u;
            __syncthreads();
#pragma unroll
            for (uint32_t q = 0; q < PER; ++q)
                if (q * T + tid < E)
                    atomicAdd(&cur[pos[q] >> 1], 1u << ((pos[q] & 1u) * 16u));
            __syncthreads();
            // cur[p] = first slot of position p's list; a wave scans its
            // share of the words, 64 at a time
            {
                const uint32_t chunk = ((words + WAVES - 1u) / WAVES + 63u) & ~63u;
                const uint32_t w0 = min(wave * chunk, words), w1 = min(w0 + chunk, words);
                uint32_t tot = 0;
                for (uint32_t w = w0 + lane; w < w1; w += 64u)
                    tot += (cur[w] & 0xFFFFu) + (cur[w] >> 16);
                tot = read_lane(wave_scan_add(tot), 63u);
                if (lane == 0u)
                    wsum[wave] = tot;
                __syncthreads();
                uint32_t carry = 0;
                for (uint32_t w = 0; w < wave; ++w)
                    carry += wsum[w];
                for (uint32_t c = w0; c < w1; c += 64u) {
                    const uint32_t w = c + lane;
                    const uint32_t x = w < w1 ? cur[w] : 0u;
                    const uint32_t pair = (x & 0xFFFFu) + (x >> 16);
                    const uint32_t inc = wave_scan_add(pair);
                    const uint32_t a0 = carry + inc - pair;
                    if (w < w1)
                        cur[w] = a0 | ((a0 + (x & 0xFFFFu)) << 16);
                    carry += read_lane(inc, 63u);
                }
            }
            __syncthreads();
#pragma unroll
            for (uint32_t q = 0; q < PER; ++q)
                if (q * T + tid < E) {
                    const uint32_t sh = (pos[q] & 1u) * 16u;
                    const uint32_t at = (atomicAdd(&cur[pos[q] >> 1], 1u << sh) >> sh) & 0xFFFFu;
                    list[at] = step[q];
                }
            __syncthreads();
            // successors, and F where the step is its list's smallest (all
            // ones: none, or not the smallest): the cursor of p is now the
            // end of its list, and p + 1's list starts there
            auto half = [&](uint32_t p) { return (cur[p >> 1] >> ((p & 1u) * 16u)) & 0xFFFFu; };
#pragma unroll
            for (uint32_t q = 0; q < PER; ++q) {
                succ[q] = first[q] = 0xFFFFFFFFu;
                if (q * T + tid < E) {
                    const uint32_t p = pos[q];
                    bool below;
                    succ[q] = rsb_list_scan(list, p ? half(p - 1u) : 0u, half(p), step[q], below);
                    if (!below)
                        first[q] = step[q] > lo + p ? step[q] : succ[q];
                }
            }
            __syncthreads();
            for (uint32_t j = tid; j < W; j += T)
                list[j] = DONE | (lo + j);
            __syncthreads();
#pragma unroll
            for (uint32_t q = 0; q < PER; ++q)
                if (first[q] != 0xFFFFFFFFu)
                    list[pos[q]] = first[q] >= hi ? DONE | V[first[q]] : first[q] - lo;
            // pointer jumping to the ends of the chains inside the bucket
            for (;;) {
                __syncthreads();
                bool open = false;
                for (uint32_t j = tid; j < W; j += T) {
                    const uint32_t v = list[j];
                    if (!(v & DONE)) {
                        const uint32_t nv = list[v];
                        list[j] = nv;
                        open |= !(nv & DONE);
                    }
                }
                if (!__syncthreads_or(open))
                    break;
            }
            for (uint32_t j = tid; j < W; j += T)
                V[lo + j] = list[j] & ~DONE;
            if (b == 0u && tid == 0u)
                row[0] = (int32_t)(list[0] & ~DONE);
#pragma unroll
            for (uint32_t q = 0; q < PER; ++q)
                if (q * T + tid < E) {
                    const uint32_t s = succ[q];
                    row[step[q]] = (int32_t)(s == 0xFFFFFFFFu ? lo + pos[q]
                                             : s >= hi        ? V[s]
                                                              : list[s - lo] & ~DONE);
                }
            __threadfence_block();
            __syncthreads();
        }
    }
}

static size_t rs_apply_lds_bytes(uint32_t n)
{
    return (size_t)((n + 2u) / 2u) * 4u + (((size_t)n * 2u + 3u) & ~(size_t)3u);
}

// ---------------------------------------------------------------------------
// Union-find state.  A node's code is either its parent's index (non-root)
// or, for a root, the cluster size and which spanning side (0 none, 1 first,
// 2 second) the cluster touches.  Touching both sides is recorded once as
// the run's spanning step and not stored (spanning is monotone).
// ---------------------------------------------------------------------------

// 16-bit codes in LDS for N <= 16384, with P = 2^shift the least power of
// two >= N: c < N parent; c >= P root with c = (1 + f) * P + (size - 1).
// The largest code, 4P - 1, fits 16 bits; decoding is a shift and a mask
// (the resolver's rounds are bound by the instructions they issue).
struct LdsState {
    static constexpr bool LDS = true;
    uint16_t *code;
    uint32_t P, shift;
    __device__ __forceinline__ uint32_t get(uint32_t i) const { return code[i]; }
    __device__ __forceinline__ void set(uint32_t i, uint32_t v) const { code[i] = (uint16_t)v; }
    __device__ __forceinline__ bool is_root(uint32_t v) const { return v >= P; }
    __device__ __forceinline__ uint32_t root(uint32_t size, uint32_t f) const { return ((1u + f) << shift) + size - 1u; }
    // LDS operations of one wavefront complete in order
    __device__ __forceinline__ void sync() const {}
    __device__ __forceinline__ void decode(uint32_t v, uint32_t &size, uint32_t &f) const
    {
        f = (v >> shift) - 1u;
        size = (v & (P - 1u)) + 1u;
    }
};

// 32-bit codes in HBM for larger N: bit 31 marks a root, bits 29-30 the
// side, bits 0-28 the size.
struct GlobalState {
    static constexpr bool LDS = false;
    uint32_t *code;
    __device__ __forceinline__ uint32_t get(uint32_t i) const { return code[i]; }
    __device__ __forceinline__ void set(uint32_t i, uint32_t v) const { code[i] = v; }
    __device__ __forceinline__ bool is_root(uint32_t v) const { return (v >> 31) != 0u; }
    __device__ __forceinline__ uint32_t root(uint32_t size, uint32_t f) const { return 0x80000000u | (f << 29) | size; }
    // stores of some lanes must be visible to loads of others
    __device__ __forceinline__ void sync() const { __threadfence_block(); }
    __device__ __forceinline__ void decode(uint32_t v, uint32_t &size, uint32_t &f) const
    {
        size = v & 0x1FFFFFFFu;
        f = (v >> 29) & 3u;
    }
};

template <typename RecT>
__device__ __forceinline__ RecT pack_record(uint32_t a, uint32_t b);
template <>
__device__ __forceinline__ uint32_t pack_record<uint32_t>(uint32_t a, uint32_t b) { return a | (b << 16); }
template <>
__device__ __forceinline__ uint64_t pack_record<uint64_t>(uint32_t a, uint32_t b) { return (uint64_t)a | ((uint64_t)b << 32); }

__device__ __forceinline__ void unpack_record(uint32_t r, uint32_t &a, uint32_t &b)
{
    a = r & 0xFFFFu;
    b = r >> 16;
}
__device__ __forceinline__ void unpack_record(uint64_t r, uint32_t &a, uint32_t &b)
{
    a = (uint32_t)r;
    b = (uint32_t)(r >> 32);
}

// The HBM-state loop of find2, from codes cx, cy already read (rx, ry:
// whether they are root codes): path halving until both are roots.
template <class St>
__device__ __forceinline__ void follow2(const St &st, uint32_t &x, uint32_t &cx, bool rx,
                                        uint32_t &y, uint32_t &cy, bool ry)
{
    while (!(rx && ry)) {
        const uint32_t gx = rx ? cx : st.get(cx);
        const uint32_t gy = ry ? cy : st.get(cy);
        if (!rx) {
            if (st.is_root(gx)) {
                x = cx;
                cx = gx;
                rx = true;
            } else {
                st.set(x, gx);
                x = gx;
                cx = st.get(x);
                rx = st.is_root(cx);
            }
        }
        if (!ry) {
            if (st.is_root(gy)) {
                y = cy;
                cy = gy;
                ry = true;
            } else {
                st.set(y, gy);
                y = gy;
                cy = st.get(y);
                ry = st.is_root(cy);
            }
        }
    }
}

// Two interleaved finds with path halving.  Concurrent halving by other
// lanes of the wave only ever replaces a parent by an ancestor, so every
// lane still reaches its true root.  With the state in LDS each pass is
// branch-free: both grandparents are read together, then (after the
// halving stores) both new nodes' codes, so a pass is two LDS round trips
// and about half the instructions of a branch per element (which also
// waits for each read in turn).  A finished element re-reads its own node,
// which costs nothing in LDS; in HBM those reads would be traffic, so the
// global state keeps the branches.
template <class St>
__device__ __forceinline__ void find2(const St &st, uint32_t &x, uint32_t &cx,
                                      uint32_t &y, uint32_t &cy)
{
    cx = st.get(x);
    cy = st.get(y);
    bool rx = st.is_root(cx), ry = st.is_root(cy);
    if constexpr (St::LDS) {
        while (!(rx && ry)) {
            const uint32_t gx = st.get(rx ? x : cx);
            const uint32_t gy = st.get(ry ? y : cy);
            const bool gxr = st.is_root(gx), gyr = st.is_root(gy);
            if (!rx && !gxr)
                st.set(x, gx);
            if (!ry && !gyr)
                st.set(y, gy);
            x = rx ? x : (gxr ? cx : gx);
            y = ry ? y : (gyr ? cy : gy);
            const uint32_t nx = st.get(x), ny = st.get(y);
            cx = rx ? cx : nx;
            cy = ry ? cy : ny;
            rx = st.is_root(cx);
            ry = st.is_root(cy);
        }
        return;
    }
    follow2(st, x, cx, rx, y, cy, ry);
}

// ---------------------------------------------------------------------------
// Merge-record arithmetic.  WIDE (N > 16384) keeps S3, S4 and the moments in
// 128 bits; otherwise every Sk fits 64 bits (Sk <= N**k <= 2**56).
// ---------------------------------------------------------------------------
template <bool WIDE>
struct Wide {
    using T = typename std::conditional<WIDE, u128, uint64_t>::type;
};

template <bool WIDE>
struct Deltas {
    using MT = typename Wide<WIDE>::T;
    using D2 = typename std::conditional<WIDE, uint64_t, uint32_t>::type;
    uint32_t dmax; // size s of the merged cluster (0: no merge)
    D2 d2;         // s^2 - a^2 - b^2 = 2 q, q = a b
    MT d3, d4;     // s^3 - a^3 - b^3 = 3 q s, s^4 - a^4 - b^4 = 2 q (2 s^2 - q)
    template <typename RecT>
    __device__ __forceinline__ explicit Deltas(RecT rec)
    {
        uint32_t a, b;
        unpack_record(rec, a, b);
        const uint32_t s = a + b;
        dmax = s;   // a record without a merge is 0
        if constexpr (WIDE) {
            // s <= 2^28
            const uint64_t q = (uint64_t)a * b;
            d2 = 2u * q;
            d3 = (MT)q * (MT)(3u * s);
            d4 = (MT)(2u * q) * (MT)(2u * ((uint64_t)s * s) - q);
        } else {
            // s <= 2^14: full-rate 24-bit products below 2^28
            const uint32_t q = (uint32_t)__umul24(a, b);
            d2 = 2u * q;
            d3 = (uint64_t)q * (3u * s);
            d4 = (uint64_t)(2u * q) * (2u * (uint32_t)__umul24(s, s) - q);
        }
    }
    __device__ __forceinline__ bool merge() const { return dmax != 0u; }
};

// Word w of a chunk-state entry: {max cluster size, merges, S2, S3 lo,
// S3 hi, S4 lo, S4 hi, 0}.
template <typename MT>
__device__ __forceinline__ uint64_t state_word(uint32_t w, uint64_t mx,
                                               uint64_t merges, uint64_t s2,
                                               MT s3, MT s4)
{
    switch (w) {
    case 0: return mx;
    case 1: return merges;
    case 2: return s2;
    case 3: return (uint64_t)s3;
    case 4: return (uint64_t)((u128)s3 >> 64);
    case 5: return (uint64_t)s4;
    case 6: return (uint64_t)((u128)s4 >> 64);
    default: return 0u;
    }
}

// Puts a uniform value into one lane (a compare and a select, no branch).
template <typename T>
__device__ __forceinline__ T write_lane(T v, uint32_t lane, T old)
{
    return threadIdx.x == lane ? v : old;
}

// Conflict table for the parallel merge rounds: CLAIM_SLOTS words in LDS,
// indexed by a multiplicative hash of a root's low 24 bits (a full-rate
// 24-bit multiply; a collision only blocks a merge for a round).
#define CLAIM_BITS 10
#define CLAIM_SLOTS (1u << CLAIM_BITS)

__device__ __forceinline__ uint32_t claim_slot(uint32_t root)
{
    return ((root & 0xFFFFFFu) * 0x9E3779u) >> (32 - CLAIM_BITS);
}

// Modified-root stamps of an HBM-state sweep: DIRTY_SLOTS words in LDS,
// indexed by the same kind of hash; a slot holds 1 + the last batch in
// which the resolver changed a root hashing there (0: never).  Collisions
// only make a root look changed.
#define DIRTY_BITS 11
#define DIRTY_SLOTS (1u << DIRTY_BITS)

__device__ __forceinline__ uint32_t dirty_slot(uint32_t root)
{
    return ((root & 0xFFFFFFu) * 0x9E3779u) >> (32 - DIRTY_BITS);
}

// One run on one wavefront.  Bonds are taken 64 at a time (lane = step):
//  1. every lane finds the roots of its bond's endpoints in parallel (path
//     halving); lanes whose roots differ are candidate merges;
//  2. parallel rounds: each candidate claims the table slots of its two
//     roots with an atomic max of (round tag + 63 - lane), so each slot ends
//     up held by the earliest candidate touching it.  A candidate holding
//     both of its slots shares no root with any earlier pending candidate:
//     no earlier merge can change its clusters, so it merges now, in
//     parallel with the other such candidates (their roots are distinct).
//     Star merges: the root the first blocked candidate is blocked on (the
//     hub, near and above the threshold usually the largest cluster's root)
//     takes in, in the same round, every pending candidate touching it, in
//     step order up to the first whose other root an earlier candidate also
//     touches, and up to the first other pending candidate that touches a
//     root the star absorbs; their records follow from an exclusive prefix
//     sum of the absorbed sizes and the spanning step from two flag
//     ballots.  The
//     others re-find their roots and go to the next round; the rounds stop
//     early once one frees at most a single candidate.  Hash collisions
//     only make the tests conservative;
//  3. the candidates left after `rounds` rounds are resolved in step order
//     with uniform control flow: roots re-read from the state (one address
//     for the whole wave, made uniform with readfirstlane) and followed
//     while earlier merges moved them, the union decided on scalar
//     registers, lane 0 writing it back, the record placed with a lane
//     select.
// Per-step output is one merge record; the spanning step is kept scalar.
// With chunk_out, the run's state at the start of every batch of 64 bonds
// (the chunk state of chunk_scan) is written as well: the batch's records
// are in registers at its end, so their deltas are reduced across the wave
// there and no pass over the records is needed.
// SPLIT (two wavefronts per run): wave 1, the finder, runs step 1 for batch
// b + 1 while wave 0, the resolver, runs steps 2 and 3 for batch b; one
// barrier per batch, the roots handed over through LDS.  A find that runs
// beside the merges of batch b may stop at a root linked meanwhile, which is
// still an ancestor: the resolver's find continues from it, usually with a
// single read.  With chunk_out and the state in LDS, the finder folds the
// records of batch b - 1 into the running state, off the resolver's chain;
// with the state in HBM the finder's dependent reads set the pace, so the
// resolver folds its own records in the time it would wait.  With the state
// in HBM the finder also hands over the code (size and sides) of each root
// it found, and the resolver stamps every root it changes with the batch in
// an LDS table (hashed, so a collision only costs a read): a handed root
// whose stamp is older than the batch the finder ran beside has not changed
// since the finder read it, so the resolver takes it without a read.
// Edge sources of the sweep: edge e -> its endpoints (u, v).
// EdgeList reads the graph's edge array.  LatticeEdges computes them for the
// square lattice of side L in the order square_lattice builds (rows r =
// 0..L-1; in each row but the last, node (r, c)'s edge to (r + 1, c), then
// to (r, c + 1) when c < L - 1; the last row's L - 1 edges to the right),
// with node (r, c) stored at r L + c, or, tiled (L a multiple of 8), in
// 4 x 8 tiles of one 128-byte line each: ((r / 4) (L / 8) + c / 8) 32 +
// (r mod 4) 8 + c mod 8, the order of the host's locality relabelling.  No
// memory is read for an edge.
struct EdgeList {
    const int2 *__restrict__ p;
    __device__ __forceinline__ int2 operator()(int32_t e) const { return p[e]; }
};

struct LatticeEdges {
    uint32_t L, d;   // side, edges per row but the last (2 L - 1)
    float inv_d;     // 1 / d, a first guess of the row
    uint32_t tiled;
    __device__ __forceinline__ uint32_t node(uint32_t r, uint32_t c) const
    {
        return tiled ? ((((r >> 2) * (L >> 3) + (c >> 3)) << 5) | ((r & 3u) << 3) | (c & 7u))
                     : r * L + c;
    }
    // bond x: its first node (r, c), and whether it goes down or to the right
    __device__ __forceinline__ void bond(uint32_t x, uint32_t &r, uint32_t &c,
                                         uint32_t &down) const
    {
        r = (uint32_t)((float)x * inv_d);
        // the float guess is off by at most one row either way
        if (r * d > x)
            --r;
        else if ((r + 1u) * d <= x)
            ++r;
        const uint32_t q = x - r * d;
        const bool last = r + 1u >= L;   // the last row: to the right only
        c = last ? q : q >> 1;
        down = last ? 0u : (~q & 1u);
    }
    __device__ __forceinline__ int2 operator()(int32_t e) const
    {
        uint32_t r, c, down;
        bond((uint32_t)e, r, c, down);
        return make_int2((int32_t)node(r, c), (int32_t)node(r + down, c + 1u - down));
    }
};

template <class St, typename RecT, bool CHUNKS, bool SPLIT, class ES, bool FOLDER = false>
__device__ __forceinline__ void sweep_run(const St &st, uint32_t N, uint32_t M,
                                          const ES &edges,
                                          const uint8_t *__restrict__ sides,
                                          bool span_first, uint32_t rounds,
                                          uint32_t *__restrict__ claims,
                                          uint32_t *__restrict__ handoff,
                                          uint32_t *__restrict__ dirty,
                                          const int32_t *__restrict__ perm,
                                          RecT *__restrict__ rec_out,
                                          uint32_t *__restrict__ span_out,
                                          uint64_t *__restrict__ chunk_out)
{
    // the sweep's pace is the resolver's dependent instruction chain: let
    // its waves win instruction arbitration over waves of other kernels
    // sharing the SIMD (the reductions of the previous sub-batch run beside
    // it).  The finder keeps the same priority: lowering it measured slower.
    __builtin_amdgcn_s_setprio(3);
    // HBM-state graphs (N > 16384) need 128-bit S3 and S4
    constexpr bool WIDE = std::is_same<St, GlobalState>::value;
    using MT = typename Wide<WIDE>::T;
    constexpr uint32_t THREADS = SPLIT ? (FOLDER ? 192u : 128u) : 64u;
    // who folds the records into the chunk states: with the state in LDS
    // the finder (the resolver sets the pace); with the state in HBM a third
    // wave (FOLDER), or else the resolver
    static_assert(!FOLDER || (SPLIT && CHUNKS && std::is_same<St, GlobalState>::value),
                  "a folder wave only for chunk states with the state in HBM");
    constexpr bool RES_FOLD = SPLIT && WIDE && !FOLDER;
    // HBM state with a finder: the finder hands over the codes of the roots
    // it found as well (after the two root slots), and the resolver reads a
    // root afresh only if, in the batch before (beside which the finder
    // read it), it changed a root hashing to the same stamp slot
    constexpr bool HANDED = SPLIT && WIDE;
    uint32_t *const codes_out = handoff + 256u;
    const uint32_t lane = threadIdx.x % 64u;
    // SPLIT: wave 0 resolves batch b while wave 1 finds the roots of batch
    // b + 1 (a find that runs beside the merges of batch b may stop at a
    // root linked meanwhile; that is still an ancestor, and the resolver's
    // find continues from it)
    const bool resolver = !SPLIT || threadIdx.x < 64u;
    const bool folder = FOLDER && threadIdx.x >= 128u;
    uint64_t cs_mx = 1, cs_merges = 0, cs_s2 = N;
    MT cs_s3 = N, cs_s4 = N;
    for (uint32_t i = threadIdx.x; i < N; i += THREADS)
        st.set(i, st.root(1u, sides ? (uint32_t)sides[i] : 0u));
    for (uint32_t i = threadIdx.x; i < CLAIM_SLOTS; i += THREADS)
        claims[i] = 0u;
    if (HANDED)
        for (uint32_t i = threadIdx.x; i < DIRTY_SLOTS; i += THREADS)
            dirty[i] = 0u;
    __syncthreads();

    uint32_t span_at = PC_NO_SPAN;
    uint32_t tag = 0;

    // one wavefront per run: the permutation two batches ahead and the edge
    // endpoints one batch ahead are in flight while a batch is resolved
    int32_t e_ahead = 0;
    int2 uv_next = make_int2(0, 0);
    if (!SPLIT) {
        e_ahead = (64u + lane < M) ? perm[64u + lane] : 0;
        if (lane < M)
            uv_next = edges(perm[lane]);
    }
    // codes of the next batch's endpoints, read one batch early: parent
    // links only ever move up the tree (a union links a root under a root,
    // halving replaces a parent by its grandparent), so a code read before
    // this batch's merges still names an ancestor and the next find may
    // start there, one dependent read shorter.  A root code is no hint
    // (the node may have been linked since): that find reads afresh.
    uint32_t hint_u = 0xFFFFFFFFu, hint_v = 0xFFFFFFFFu;

    // SPLIT finder: roots of the batch at b0 into handoff slot (b0 / 64) & 1
    // (u roots in words 0..63, v roots in 64..127 of the slot).  Its own
    // pipeline, issued at the start of a batch so the loads complete beside
    // the finds: the permutation three batches ahead, the endpoints two
    // batches ahead, and the codes of the next batch's endpoints (the hints
    // above; with the state in HBM the finder is the slower wave and each
    // hint saves a dependent read)
    int2 f_uv1 = make_int2(0, 0), f_uv2 = make_int2(0, 0);
    int32_t f_e3 = 0;
    uint32_t f_hu = 0xFFFFFFFFu, f_hv = 0xFFFFFFFFu;
    if (SPLIT && !resolver && !folder) {
        if (lane < M)
            f_uv1 = edges(perm[lane]);
        if (64u + lane < M)
            f_uv2 = edges(perm[64u + lane]);
        f_e3 = (128u + lane < M) ? perm[128u + lane] : 0;
    }
    auto find_batch = [&](uint32_t b0) {
        const int2 uv = f_uv1;
        const uint32_t hu = f_hu, hv = f_hv;
        f_uv1 = f_uv2;
        if (b0 + 64u + lane < M) {
            f_hu = st.get((uint32_t)f_uv1.x);
            f_hv = st.get((uint32_t)f_uv1.y);
        }
        f_uv2 = (b0 + 128u + lane < M) ? edges(f_e3) : make_int2(0, 0);
        f_e3 = (b0 + 192u + lane < M) ? perm[b0 + 192u + lane] : 0;
        uint32_t x = st.is_root(hu) ? (uint32_t)uv.x : hu;
        uint32_t y = st.is_root(hv) ? (uint32_t)uv.y : hv;
        uint32_t cx, cy;
        if (HANDED)
            cx = cy = st.root(1u, 0u);   // a root code on idle lanes
        if (b0 + lane < M)
            find2(st, x, cx, y, cy);
        const uint32_t si = ((b0 / 64u) & 1u) * 128u;
        handoff[si + lane] = x;
        handoff[si + 64u + lane] = y;
        if (HANDED) {
            codes_out[si + lane] = cx;
            codes_out[si + 64u + lane] = cy;
        }
    };
    if (SPLIT) {
        if (!resolver && !folder)
            find_batch(0u);
        __syncthreads();
    }

    // SPLIT with chunk states: the resolver hands each batch's records to
    // the wave that folds them (two slots of 64 records after the root
    // slots, after the roots' codes with the state in HBM), which folds them
    // into the running state one batch later, off the resolver's chain
    RecT *rec_slots = (RecT *)(handoff + (HANDED ? 512u : 256u));
    auto fold_batch = [&](RecT rec) {
        Deltas<WIDE> d(rec);
        cs_merges += (uint32_t)__popcll(ballot(d.merge()));
        scan_state(d.dmax, d.d2, d.d3, d.d4);
        cs_mx = umax64(cs_mx, (uint64_t)read_lane(d.dmax, 63u));
        cs_s2 += read_lane(d.d2, 63u);
        cs_s3 += read_lane(d.d3, 63u);
        cs_s4 += read_lane(d.d4, 63u);
    };

    for (uint32_t base = 0; base < M; base += 64u) {
        if (SPLIT && !resolver) {
            if (CHUNKS && !RES_FOLD && (folder || !FOLDER)) {
                // state at the start of this batch: fold the records the
                // resolver finished in the previous iteration
                if (base > 0u)
                    fold_batch(rec_slots[(((base / 64u) - 1u) & 1u) * 64u + lane]);
                if (lane < PC_STATE_WORDS)
                    chunk_out[(size_t)(base / 64u) * PC_STATE_WORDS + lane] =
                        state_word(lane, cs_mx, cs_merges, cs_s2, cs_s3, cs_s4);
            }
            if (!folder && base + 64u < M)
                find_batch(base + 64u);
            __syncthreads();
            continue;
        }
        const uint32_t n = base + lane;
        const bool active = n < M;
        if ((!SPLIT || RES_FOLD) && CHUNKS && lane < PC_STATE_WORDS)
            chunk_out[(size_t)(base / 64u) * PC_STATE_WORDS + lane] =
                state_word(lane, cs_mx, cs_merges, cs_s2, cs_s3, cs_s4);
        uint32_t ru, rv, cu, cv;
        if (SPLIT) {
            // the finder's roots, followed past the previous batch's merges
            const uint32_t si = ((base / 64u) & 1u) * 128u;
            ru = handoff[si + lane];
            rv = handoff[si + 64u + lane];
            if (HANDED) {
                // a root unchanged since the finder read it is still a root
                // with that code: no read
                const uint32_t b = base / 64u;
                cu = codes_out[si + lane];
                cv = codes_out[si + 64u + lane];
                if (dirty[dirty_slot(ru)] >= b)
                    cu = st.get(ru);
                if (dirty[dirty_slot(rv)] >= b)
                    cv = st.get(rv);
                follow2(st, ru, cu, st.is_root(cu), rv, cv, st.is_root(cv));
            } else {
                find2(st, ru, cu, rv, cv);
            }
        } else {
            const int2 uv = uv_next;
            uv_next = (n + 64u < M) ? edges(e_ahead) : make_int2(0, 0);
            e_ahead = (n + 128u < M) ? perm[n + 128u] : 0;
            ru = st.is_root(hint_u) ? (uint32_t)uv.x : hint_u;
            rv = st.is_root(hint_v) ? (uint32_t)uv.y : hint_v;
            find2(st, ru, cu, rv, cv);
            hint_u = st.get((uint32_t)uv_next.x);
            hint_v = st.get((uint32_t)uv_next.y);
        }
        bool cand = active && ru != rv;
        uint64_t pending = ballot(cand);
        RecT rec = 0;

        if (tag >= 0xFFFFFFFFu - 65u * 64u) {
            // this batch's round tags (at most 64 rounds) could wrap: clear
            // the table and restart
            for (uint32_t i = lane; i < CLAIM_SLOTS; i += 64u)
                claims[i] = 0u;
            tag = 0u;
        }
        for (uint32_t k = 0; k < rounds && pending; ++k) {
            tag += 64u;
            const uint32_t mine = tag + 63u - lane;
            const uint32_t su = claim_slot(ru), sv = claim_slot(rv);
            if (cand) {
                atomicMax(&claims[su], mine);
                atomicMax(&claims[sv], mine);
            }
            const uint32_t held_u = claims[su], held_v = claims[sv];
            const bool own_u = held_u == mine, own_v = held_v == mine;
            bool go = cand && own_u && own_v;
            // star: the pending candidates that touch one hub root (the root
            // the first blocked candidate is blocked on, usually the largest
            // cluster's), in step order up to the first whose other root an
            // earlier candidate also touches, all merge into the hub now
            uint64_t star = 0;
            uint32_t hub = 0;
            const uint64_t blocked = ballot(cand && !go);
            if (blocked) {
                const uint32_t fl = (uint32_t)__builtin_ctzll(blocked);
                hub = read_lane(own_u ? rv : ru, fl);
                const bool at_u = ru == hub;
                const bool touch = cand && (at_u || rv == hub);
                const uint64_t tm = ballot(touch);
                const uint64_t bad = tm & ~ballot(touch && (at_u ? own_v : own_u));
                star = bad ? (tm & ((bad & (0u - bad)) - 1u)) : tm;
                go = go && !touch;
                // a pending candidate outside the star whose root's slot is
                // held by a member touches a root the star absorbs before
                // its step: the star stops before it (the slot holder is
                // the earliest claimant, lane tag + 63 - claims[slot])
                const uint32_t hu = tag + 63u - held_u, hv = tag + 63u - held_v;
                const bool late = cand && !go && !((star >> lane) & 1u) &&
                                  (((star >> (hu & 63u)) & 1u) || ((star >> (hv & 63u)) & 1u));
                const uint64_t lm = ballot(late);
                if (lm)
                    star &= (lm & (0u - lm)) - 1u;
            }
            const bool in_star = (star >> lane) & 1u;
            const uint64_t freed = ballot(go) | star;
            if (star) {
                // records in step order: the hub's size grows by the sizes
                // absorbed by the earlier members (exclusive prefix sum)
                const bool at_u = ru == hub;
                const uint32_t x = at_u ? rv : ru;
                uint32_t sx, fx, sh, fh;
                st.decode(at_u ? cv : cu, sx, fx);
                st.decode(at_u ? cu : cv, sh, fh);
                const uint32_t first = (uint32_t)__builtin_ctzll(star);
                const uint32_t s_hub = read_lane(sh, first), f_hub = read_lane(fh, first);
                const uint32_t incl = wave_scan_add(in_star ? sx : 0u);
                const uint32_t total = read_lane(incl, 63u);
                const uint64_t m1 = ballot(in_star && (fx & 1u));
                const uint64_t m2 = ballot(in_star && (fx & 2u));
                const uint32_t f_all = f_hub | (m1 ? 1u : 0u) | (m2 ? 2u : 0u);
                if (in_star) {
                    // (size on u's side, size on v's side), as every merge
                    st.set(x, hub);
                    if (HANDED)
                        dirty[dirty_slot(x)] = base / 64u + 1u;
                    const uint32_t sh_now = s_hub + incl - sx;
                    rec = pack_record<RecT>(at_u ? sh_now : sx, at_u ? sx : sh_now);
                }
                if (lane == first) {
                    st.set(hub, st.root(s_hub + total, f_all == 3u ? 0u : f_all));
                    if (HANDED)
                        dirty[dirty_slot(hub)] = base / 64u + 1u;
                }
                if (span_first)
                    span_at = min(span_at, base + first + 1u);
                if (f_all == 3u) {
                    // first member after which both sides are touched
                    const uint32_t l1 = (f_hub & 1u) ? first : (uint32_t)__builtin_ctzll(m1);
                    const uint32_t l2 = (f_hub & 2u) ? first : (uint32_t)__builtin_ctzll(m2);
                    span_at = min(span_at, base + max(l1, l2) + 1u);
                }
            }
            bool spans_here = false;
            if (go) {
                uint32_t sa, fa, sb, fb;
                st.decode(cu, sa, fa);
                st.decode(cv, sb, fb);
                const bool a_big = sa >= sb;
                const uint32_t big = a_big ? ru : rv, small = a_big ? rv : ru;
                uint32_t f = fa | fb;
                st.set(small, big);
                st.set(big, st.root(sa + sb, f == 3u ? 0u : f));
                if (HANDED) {
                    dirty[dirty_slot(small)] = base / 64u + 1u;
                    dirty[dirty_slot(big)] = base / 64u + 1u;
                }
                rec = pack_record<RecT>(sa, sb);
                spans_here = span_first || f == 3u;
            }
            {
                const uint64_t spans = ballot(spans_here);
                if (spans)
                    span_at = min(span_at, base + (uint32_t)__builtin_ctzll(spans) + 1u);
            }
            cand = cand && !go && !in_star;
            st.sync();
            if (ballot(cand)) {
                // lanes still pending follow their roots past this round's merges
                if (cand)
                    find2(st, ru, cu, rv, cv);
                cand = cand && ru != rv;
            }
            pending = ballot(cand);
            // a round that frees at most one candidate is resolving a chain
            // (typically through the largest cluster's root): the in-order
            // remainder does that more cheaply
            if (__builtin_popcountll(freed) <= 1)
                break;
        }

        while (pending) {
            const uint32_t i = (uint32_t)__builtin_ctzll(pending);
            pending &= pending - 1u;
            uint32_t a = read_lane(ru, i), b = read_lane(rv, i);
            uint32_t ca = uniform(st.get(a)), cb = uniform(st.get(b));
            while (!st.is_root(ca)) {
                a = ca;
                ca = uniform(st.get(a));
            }
            while (!st.is_root(cb)) {
                b = cb;
                cb = uniform(st.get(b));
            }
            if (a == b)
                continue; // joined by an earlier bond of this batch
            uint32_t sa, fa, sb, fb;
            st.decode(ca, sa, fa);
            st.decode(cb, sb, fb);
            const bool a_big = sa >= sb;
            const uint32_t big = a_big ? a : b, small = a_big ? b : a;
            uint32_t f = fa | fb;
            if (f == 3u || span_first)
                span_at = min(span_at, base + i + 1u);
            if (f == 3u)
                f = 0u;
            if (lane == 0) {
                st.set(small, big);
                st.set(big, st.root(sa + sb, f));
                if (HANDED) {
                    dirty[dirty_slot(small)] = base / 64u + 1u;
                    dirty[dirty_slot(big)] = base / 64u + 1u;
                }
            }
            rec = write_lane(pack_record<RecT>(sa, sb), i, rec);
        }
        if (active)
            rec_out[n] = rec;
        if (SPLIT && CHUNKS && !RES_FOLD)
            rec_slots[((base / 64u) & 1u) * 64u + lane] = rec;
        else if (CHUNKS)
            fold_batch(rec);
        if (!SPLIT)
            __syncthreads();
        else {
            st.sync();
            __syncthreads();
        }
    }
    if (threadIdx.x == 0)
        *span_out = span_at;
}

// Words of LDS before the 16-bit codes: the claim table, then (SPLIT) the
// handoff: two slots of 128 roots, then two slots of 64 records (up to 64
// bits each; with the state in HBM, two slots of the roots' 128 codes).
#define SWEEP_HANDOFF_WORDS 512u
template <bool SPLIT>
constexpr uint32_t sweep_lds_words() { return CLAIM_SLOTS + (SPLIT ? SWEEP_HANDOFF_WORDS : 0u); }

template <typename RecT, bool CHUNKS, bool SPLIT, class ES>
__global__ __launch_bounds__(SPLIT ? 128 : 64) void sweep_lds_kernel(
    uint32_t N, uint32_t M, ES edges,
    const uint8_t *__restrict__ sides, int span_first,
    const int32_t *__restrict__ perm, int64_t perm_stride,
    RecT *__restrict__ records, int64_t rec_stride,
    uint32_t *__restrict__ span_step, uint32_t rounds,
    uint64_t *__restrict__ chunk_state)
{
    // claim table first (word aligned), the handoff slots, then the codes
    extern __shared__ uint32_t lds_words[];
    const uint32_t r = blockIdx.x;
    const size_t cstride = (size_t)((M + 63u) / 64u) * PC_STATE_WORDS;
    const uint32_t shift = N > 1u ? 32u - (uint32_t)__builtin_clz(N - 1u) : 0u;
    const LdsState st{(uint16_t *)(lds_words + sweep_lds_words<SPLIT>()), 1u << shift, shift};
    sweep_run<LdsState, RecT, CHUNKS, SPLIT, ES>(
        st, N, M, edges, sides, span_first != 0, rounds, lds_words,
        lds_words + CLAIM_SLOTS, nullptr, perm + (int64_t)r * perm_stride,
        records + (int64_t)r * rec_stride, span_step + r,
        CHUNKS ? chunk_state + r * cstride : nullptr);
}

template <typename RecT, bool CHUNKS, bool SPLIT, class ES, bool FOLDER = false>
__global__ __launch_bounds__(SPLIT ? (FOLDER ? 192 : 128) : 64) void sweep_global_kernel(
    uint32_t N, uint32_t M, uint32_t R, ES edges,
    const uint8_t *__restrict__ sides, int span_first,
    const int32_t *__restrict__ perm, int64_t perm_stride,
    RecT *__restrict__ records, int64_t rec_stride,
    uint32_t *__restrict__ span_step, uint32_t *__restrict__ workspace,
    uint32_t rounds, uint64_t *__restrict__ chunk_state,
    const uint32_t *__restrict__ only)
{
    // only: sweep the runs marked there (NULL: every run)
    // the handoff: root slots, the roots' codes, then (FOLDER) the records
    __shared__ uint32_t claims[CLAIM_SLOTS];
    __shared__ uint32_t handoff[SPLIT ? SWEEP_HANDOFF_WORDS + (FOLDER ? 256u : 0u) : 1u];
    __shared__ uint32_t dirty[SPLIT ? DIRTY_SLOTS : 1u];
    const size_t cstride = (size_t)((M + 63u) / 64u) * PC_STATE_WORDS;
    const GlobalState st{workspace + (size_t)blockIdx.x * N};
    for (uint32_t r = blockIdx.x; r < R; r += gridDim.x) {
        if (only && !only[r])
            continue;
        sweep_run<GlobalState, RecT, CHUNKS, SPLIT, ES, FOLDER>(
            st, N, M, edges, sides, span_first != 0, rounds, claims, handoff,
            dirty, perm + (int64_t)r * perm_stride, records + (int64_t)r * rec_stride,
            span_step + r, CHUNKS ? chunk_state + r * cstride : nullptr);
        __syncthreads();
    }
}

// Persistent sweep over several graphs (the lattices of a finite-size
// study) in one launch: a graph table, every graph's runs numbered in table
// order (graph g owns queue items first .. first + runs - 1), and a queue
// head in device memory.  Each workgroup takes the next item with one
// atomic, sweeps that run with the graph's state kind (LDS codes, or 32-bit
// codes in its own HBM slot), and repeats until the queue is empty, so long
// and short runs pack onto the CUs with no per-graph launch or stream.  The
// table lists the largest graphs first (their runs are the longest).  Every
// sweep folds the chunk states in the finder wave.
struct MultiGraph {
    const int2 *edges;
    LatticeEdges lattice;   // used when lattice.L != 0 (edges unused)
    const uint8_t *sides;
    const int32_t *perm;
    void *records;
    uint32_t *span_step;
    uint64_t *chunk_state;
    int64_t perm_stride, rec_stride;
    uint32_t N, M, runs, first, kind, span_first, rounds, shift;
};
#define MULTI_LDS 0u       // LDS codes, 32-bit records
#define MULTI_HBM32 1u     // HBM codes, 32-bit records
#define MULTI_HBM64 2u     // HBM codes, 64-bit records

__global__ void zero_u32_kernel(uint32_t *p) { *p = 0u; }

__global__ __launch_bounds__(128) void sweep_multi_kernel(
    const MultiGraph *__restrict__ graphs, uint32_t num_graphs, uint32_t total,
    uint32_t *__restrict__ head, uint32_t *__restrict__ workspace,
    uint64_t slot_words)
{
    extern __shared__ uint32_t lds_words[];
    __shared__ uint32_t item;
    uint32_t *claims = lds_words, *handoff = lds_words + CLAIM_SLOTS;
    // after the handoff: an LDS graph's codes, or an HBM graph's root stamps
    uint16_t *codes = (uint16_t *)(lds_words + sweep_lds_words<true>());
    uint32_t *dirty = lds_words + sweep_lds_words<true>();
    for (;;) {
        if (threadIdx.x == 0u)
            item = atomicAdd(head, 1u);
        __syncthreads();
        const uint32_t q = item;
        __syncthreads();
        if (q >= total)
            return;
        uint32_t g = 0;
        while (g + 1u < num_graphs && q >= graphs[g + 1u].first)
            ++g;
        const MultiGraph &G = graphs[g];
        const uint32_t r = q - G.first;
        const size_t cstride = (size_t)((G.M + 63u) / 64u) * PC_STATE_WORDS;
        uint64_t *cs = G.chunk_state + r * cstride;
        const int32_t *perm = G.perm + (int64_t)r * G.perm_stride;
        auto run = [&](const auto &edges) {
            if (G.kind == MULTI_LDS) {
                const LdsState st{codes, 1u << G.shift, G.shift};
                sweep_run<LdsState, uint32_t, true, true>(
                    st, G.N, G.M, edges, G.sides, G.span_first != 0u, G.rounds,
                    claims, handoff, nullptr, perm,
                    (uint32_t *)G.records + (int64_t)r * G.rec_stride,
                    G.span_step + r, cs);
            } else {
                const GlobalState st{workspace + (size_t)blockIdx.x * slot_words};
                if (G.kind == MULTI_HBM32)
                    sweep_run<GlobalState, uint32_t, true, true>(
                        st, G.N, G.M, edges, G.sides, G.span_first != 0u, G.rounds,
                        claims, handoff, dirty, perm,
                        (uint32_t *)G.records + (int64_t)r * G.rec_stride, G.span_step + r, cs);
                else
                    sweep_run<GlobalState, uint64_t, true, true>(
                        st, G.N, G.M, edges, G.sides, G.span_first != 0u, G.rounds,
                        claims, handoff, dirty, perm,
                        (uint64_t *)G.records + (int64_t)r * G.rec_stride, G.span_step + r, cs);
            }
        };
        if (G.lattice.L)
            run(G.lattice);
        else
            run(EdgeList{G.edges});
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Tiled sweep of the square lattice (pc_sweep_lattice where tile_geo takes
// it).  The lattice is cut into tiles of at
// most TILE_SIDE x TILE_SIDE nodes.  A node with a bond into another tile is
// open, and so is every cluster of a tile's own bonds that holds an open
// node; the other clusters of a tile are closed: nothing outside the tile
// can have joined them, so their sizes and sides are exact at every step.
//   1. tile_scatter: each run's bonds, in step order, into one list per
//      tile (its internal bonds); the record row, with an event for every
//      bond between two tiles and 0 elsewhere;
//   2. tile_sweep: one wavefront per (run, tile) merges the tile's internal
//      bonds in step order with its state in LDS.  A merge of two closed
//      clusters is final and its record is written.  A merge with an open
//      cluster becomes an event: the open cluster, named by one of its open
//      nodes, gains a closed cluster of known size, or joins another open
//      one.  A closed cluster goes under the open root, whose code does not
//      change, so such merges do not conflict over it: near and above the
//      threshold, where most merges hit one large cluster, a batch resolves
//      in one round;
//   3. event_sweep: one workgroup per run merges the run's events in step
//      order over the open nodes alone (0.05 N of them) and replaces every
//      event by its record.
// About 0.11 M of a random run's steps are events (64 x 64 tiles); the
// others never leave LDS.  A tile-level merge of two open clusters that
// outside bonds have already joined is found out in step 3 (record 0).
// Untiled, with every node's code in HBM, the sweep moves 342 bytes per
// addition in random lines at L = 1024, and at L = 128 (codes in LDS) four
// runs fill a CU.  Sweep with its chunk states, untiled and tiled: L = 1024,
// 1000 runs 158 and 60 ms (lists 16, tiles 19, events 20, chunk states 4);
// L = 256, 200 runs 3.67 and 1.1; L = 181, 600 runs 2.65 and 1.1; L = 128,
// 10^4 runs (no chunk states) 7.06 and 5.05.  The tiles are bound by vector
// issue (the vector ALUs are 48 % busy at L = 128, 43 % at L = 256) and
// dependent LDS round trips, and at L = 1024 by the records, which go out in
// part-written lines: rows cleared in step order by tile_scatter, so that a
// tile writes merges only, took them from 35 to 27 ms, a claim table of 512
// slots instead of 1024 (15 wavefronts per CU, not 13) to 23.  Codes that
// are addresses, a claim slot without a multiply and both claims read at once
// took 10^4 runs of L = 128 from 3.26 to 2.80 ms.
//
// Event record (half = half of a record's bits): the high half's top bit is
// set (a final record's sizes are below 2^(half - 1) on both sides in step
// 2, and step 3 reads a step before it writes it); low half: an open node's
// id; its top bit clear for a gain (high half: size, sides << 12, and bit 14
// set when the closed cluster is on the bond's u side), set for a join (high
// half: the other open node's id).
// ---------------------------------------------------------------------------
#define TILE_SIDE 64u
#define TILE_LDS_LENGTH 96u
#define TILE_MAX_LENGTH 2048u
#define TILE_CLAIM_BITS 9
#define TILE_CLAIM_SLOTS (1u << TILE_CLAIM_BITS)
#define TILE_SCATTER_BLOCKS 1024u // workgroups tile_scatter wants
// Groups of 64 steps a wave of tile_scatter takes at once: a turn of the four
// waves then gives a tile's list 1024 * groups / tiles bytes.  With eight and
// more than TILE_MANY tiles, lists and lines fill in small pieces: 16 groups
// took 1000 runs of L = 1024 (256 tiles) from 17.0 to 15.1 ms, 300 of L = 700
// (121) 2.44 to 2.27, 1000 of L = 384 (36) 1.85 to 1.70; 600 of L = 181 (9)
// 0.157 to 0.179 and 200 of L = 256 (16) 0.115 to 0.138, so fewer tiles keep
// eight, and so do segments of fewer than TILE_LONG_SEGMENT steps, where a
// turn is a large part (32 runs of L = 512, the whole sweep: 2.18 to 2.15 ms).
#define TILE_GROUPS 8u
#define TILE_GROUPS_MANY 16u
#define TILE_MANY 32u
#define TILE_LONG_SEGMENT 65536u
#define TILE_WINDOW (1u << 19)  // the steps that a list entry can tell apart

// Tiles of h x w nodes (the last row and column of tiles may be smaller),
// KH x KW of them.  mh, mw, md divide a coordinate by h and w, a bond by the
// bonds of a row (high half of the product; exact below 2^16, tile_bond
// corrects the bond's).  Ids of a tile's border nodes: per of them.
struct TileGeo {
    LatticeEdges lat;
    uint32_t L, h, w, KH, KW, K, per, mh, mw, md, init_stride;
    __host__ __device__ __forceinline__ uint32_t rows(uint32_t tr) const { return tr + 1u < KH ? h : L - (KH - 1u) * h; }
    __host__ __device__ __forceinline__ uint32_t cols(uint32_t tc) const { return tc + 1u < KW ? w : L - (KW - 1u) * w; }
    // internal bonds of a tile of hh x ww nodes, and the first list entry of
    // tile (tr, tc) when the tiles' lists follow one another
    __host__ __device__ static __forceinline__ uint32_t bonds(uint32_t hh, uint32_t ww) { return hh * (ww - 1u) + (hh - 1u) * ww; }
    __host__ __device__ __forceinline__ uint32_t offset(uint32_t tr, uint32_t tc) const
    {
        const uint32_t hh = rows(tr);
        return tr * ((KW - 1u) * bonds(h, w) + bonds(h, cols(KW - 1u))) + tc * bonds(hh, w);
    }
    __host__ __device__ __forceinline__ uint32_t bonds_of(uint32_t k) const { return bonds(rows(k / KW), cols(k % KW)); }
    // place of border node (lr, lc) of a tile of hh rows among its ids
    __device__ __forceinline__ uint32_t border(uint32_t lr, uint32_t lc, uint32_t hh) const
    {
        const uint32_t side = 2u * w + lr - 1u + (lc ? h - 2u : 0u);
        return lr == 0u ? lc : lr + 1u == hh ? w + lc : side;
    }
};

// Windows of the list entries' steps in a run of M.
__host__ __device__ __forceinline__ uint32_t tile_windows(uint32_t M) { return (M + TILE_WINDOW - 1u) / TILE_WINDOW; }

// A tile's union-find code, with nodes named by the byte offset of their code
// (twice the local index, so a code is an address): a parent's offset (below
// 0x2000), an open root's place among the tile's ids (0x2000 + place), or a
// closed root's 0x4000 | sides << 12 | size.
#define TILE_OPEN 0x2000u
#define TILE_CLOSED 0x4000u
struct TileState {
    static constexpr bool LDS = true;
    char *code;
    __device__ __forceinline__ uint32_t get(uint32_t i) const { return *(uint16_t *)(code + i); }
    __device__ __forceinline__ void set(uint32_t i, uint32_t v) const { *(uint16_t *)(code + i) = (uint16_t)v; }
    __device__ __forceinline__ bool is_root(uint32_t v) const { return v >= TILE_OPEN; }
};

template <typename RecT>
struct EventBits {
    static constexpr uint32_t half = sizeof(RecT) * 4u;
    static constexpr uint32_t top = 1u << (half - 1u);
    static __device__ __forceinline__ RecT join(uint32_t a, uint32_t b) { return pack_record<RecT>(a | top, b | top); }
    static __device__ __forceinline__ bool is_event(RecT r) { return (r >> (2u * half - 1u)) != 0; }
};

// List entries: step modulo TILE_WINDOW, local index of u (taken as its code's
// offset), and whether v is the node below u (else the one to its right).
// Where a run has more steps, tile_scatter notes how far each list has come
// at every multiple of TILE_WINDOW.  (With 64-bit entries that hold the whole
// step, 1000 runs of L = 1024 took 19.1 ms to scatter and 20.2 to sweep; with
// these 17.0 and 19.4, in two slabs of runs instead of four.)
struct TileEntry {
    static __device__ __forceinline__ uint32_t make(uint32_t t, uint32_t u, uint32_t down) { return (t & (TILE_WINDOW - 1u)) | (u << 19) | (down << 31); }
    static __device__ __forceinline__ void take(uint32_t e, uint32_t &t, uint32_t &u, uint32_t &down)
    {
        t = e & (TILE_WINDOW - 1u);
        u = (e >> 18) & 0x1FFEu;
        down = e >> 31;
    }
};

// Bond e in its tile: the tile k of its first node, that node's local row
// and column, whether the bond goes down, and whether it leaves the tile.
struct TileBond {
    uint32_t k, tr, lr, lc, down;
    bool cross;
};
__device__ __forceinline__ TileBond tile_bond(const TileGeo &g, int32_t e)
{
    // row and place in it, as LatticeEdges::bond: the high half of the product
    // with ceil(2^32 / d) is the quotient or one more, below 2^32 / d bonds
    uint32_t r = __umulhi((uint32_t)e, g.md);
    int32_t j = e - (int32_t)(r * g.lat.d);
    r -= j < 0 ? 1u : 0u;
    j += j < 0 ? (int32_t)g.lat.d : 0;
    const bool last = r + 1u == g.L;
    const uint32_t c = last ? (uint32_t)j : (uint32_t)j >> 1;
    TileBond b;
    b.down = last ? 0u : ~(uint32_t)j & 1u;
    b.tr = __umulhi(r, g.mh);
    const uint32_t tc = __umulhi(c, g.mw);
    b.lr = r - b.tr * g.h;
    b.lc = c - tc * g.w;
    b.k = b.tr * g.KW + tc;
    b.cross = (b.down ? b.lr : b.lc) + 1u == g.h;   // h = w
    return b;
}

// Initial codes of every tile's nodes and of the open nodes' own forest.
__global__ __launch_bounds__(256) void tile_init_kernel(
    TileGeo g, const uint8_t *__restrict__ sides, uint16_t *__restrict__ tiles,
    uint32_t *__restrict__ open)
{
    const uint32_t k = blockIdx.x, tr = k / g.KW, tc = k % g.KW;
    const uint32_t hh = g.rows(tr), ww = g.cols(tc);
    for (uint32_t i = threadIdx.x; i < g.per; i += 256u)
        open[k * g.per + i] = 0x80000001u;   // also the ids of no open node
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < g.init_stride; i += 256u) {
        const uint32_t lr = i / g.w, lc = i % g.w;
        uint32_t v = 0;
        if (lr < hh && lc < ww) {
            const uint32_t f = sides ? (uint32_t)sides[g.lat.node(tr * g.h + lr, tc * g.w + lc)] : 0u;
            const bool is_open = (lr == 0u && tr) || (lr + 1u == hh && tr + 1u < g.KH) ||
                                 (lc == 0u && tc) || (lc + 1u == ww && tc + 1u < g.KW);
            v = TILE_CLOSED | (f << 12) | 1u;
            if (is_open) {
                const uint32_t id = g.border(lr, lc, hh);
                v = TILE_OPEN + id;
                open[k * g.per + id] = 0x80000000u | (f << 29) | 1u;
            }
        }
        tiles[(size_t)k * g.init_stride + i] = (uint16_t)v;
    }
}

// Internal bonds per (run, segment of steps, tile), where a run's steps are
// cut into nseg segments for several workgroups.
__global__ __launch_bounds__(256) void tile_count_kernel(
    TileGeo g, uint32_t M, uint32_t seg_steps, const int32_t *__restrict__ perm,
    int64_t perm_stride, uint32_t *__restrict__ counts)
{
    extern __shared__ uint32_t tile_cnt[];
    const uint32_t seg = blockIdx.x, nseg = gridDim.x;
    for (uint32_t k = threadIdx.x; k < g.K; k += 256u)
        tile_cnt[k] = 0u;
    __syncthreads();
    const int32_t *p = perm + (int64_t)blockIdx.y * perm_stride;
    const uint32_t end = min(M, (seg + 1u) * seg_steps);
    // eight bonds a thread in flight (1000 runs of L = 1024: 2.0 ms, one at a
    // time 3.8; 500 of L = 100 17 us, 35)
    for (uint32_t t0 = seg * seg_steps + threadIdx.x; t0 < end; t0 += 8u * 256u) {
        uint32_t e[8];
#pragma unroll
        for (uint32_t i = 0; i < 8u; ++i)
            e[i] = (uint32_t)p[min(t0 + i * 256u, M - 1u)];
#pragma unroll
        for (uint32_t i = 0; i < 8u; ++i) {
            const bool ok = t0 + i * 256u < end && e[i] < M;
            const TileBond b = tile_bond(g, (int32_t)(ok ? e[i] : 0u));
            if (ok && !b.cross)
                atomicAdd(&tile_cnt[b.k], 1u);
        }
    }
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < g.K; k += 256u)
        counts[((size_t)blockIdx.y * nseg + seg) * g.K + k] = tile_cnt[k];
}

// Counts to exclusive prefixes over a run's segments; odd[run] is set when a
// tile's count is not its number of bonds.
__global__ __launch_bounds__(256) void tile_scan_kernel(
    TileGeo g, uint32_t nseg, uint32_t *__restrict__ counts, uint32_t *__restrict__ odd)
{
    uint32_t *c = counts + (size_t)blockIdx.x * nseg * g.K;
    bool wrong = false;
    for (uint32_t k = threadIdx.x; k < g.K; k += 256u) {
        uint32_t acc = 0;
        for (uint32_t s = 0; s < nseg; ++s) {
            const uint32_t n = c[(size_t)s * g.K + k];
            c[(size_t)s * g.K + k] = acc;
            acc += n;
        }
        wrong |= acc != g.bonds_of(k);
    }
    const int any = __syncthreads_or(wrong);
    if (threadIdx.x == 0u)
        odd[blockIdx.x] = any ? 1u : 0u;
}

// The tiles' lists of a run (or of one segment of its steps): a stable
// counting sort by tile of 256 * GROUPS steps at a time.  Every wave
// ranks its 64 * GROUPS consecutive steps (match_label, and the wave's
// own counter of each tile), the counters of the four waves become places
// after the tile's cursor, and the entries are stored.  A row that is not a
// permutation (some bond twice) may not fill the lists: such a run is marked
// in odd[] and left to the untiled sweep.
template <typename RecT, uint32_t GROUPS>
__global__ __launch_bounds__(256) void tile_scatter_kernel(
    TileGeo g, uint32_t M, uint32_t tile_bits, uint32_t seg_steps,
    const int32_t *__restrict__ perm, int64_t perm_stride,
    const uint32_t *__restrict__ counts, uint32_t *__restrict__ lists, int64_t list_stride,
    uint32_t *__restrict__ windows, RecT *__restrict__ records, int64_t rec_stride,
    uint32_t *__restrict__ span_step, uint32_t *__restrict__ odd)
{
    // a window starts at the start of some turn of the loop below
    static_assert(TILE_WINDOW % (256u * GROUPS) == 0u, "turns must meet the windows' starts");
    extern __shared__ uint32_t tile_dyn[];   // [4][K] wave counters, [K] cursors
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t seg = blockIdx.x, nseg = gridDim.x, run = blockIdx.y;
    uint32_t *my = tile_dyn + wave * g.K, *cursor = tile_dyn + 4u * g.K;
    for (uint32_t k = tid; k < g.K; k += 256u)
        cursor[k] = g.offset(k / g.KW, k % g.KW) +
                    (nseg > 1u ? counts[((size_t)run * nseg + seg) * g.K + k] : 0u);
    if (seg == 0u && tid == 0u)
        span_step[run] = PC_NO_SPAN;
    if (nseg > 1u && odd[run])
        return;
    bool wrong = false;
    const int32_t *p = perm + (int64_t)run * perm_stride;
    uint32_t *list = lists + (int64_t)run * list_stride;
    RecT *rec = records + (int64_t)run * rec_stride;
    const uint32_t end = min(M, (seg + 1u) * seg_steps);
    int32_t e[GROUPS];
    uint32_t t0 = seg * seg_steps + wave * 64u * GROUPS + lane;
    auto load = [&]() {
#pragma unroll
        for (uint32_t i = 0; i < GROUPS; ++i)
            e[i] = p[min(t0 + i * 64u, M - 1u)];
    };
    load();
    for (uint32_t base = seg * seg_steps; base < end; base += 256u * GROUPS) {
        for (uint32_t k = lane; k < g.K; k += 64u)
            my[k] = 0u;
        if (M > TILE_WINDOW && base % TILE_WINDOW == 0u) {
            uint32_t *to = windows + ((size_t)run * tile_windows(M) + base / TILE_WINDOW) * g.K;
            for (uint32_t k = tid; k < g.K; k += 256u)
                to[k] = cursor[k];
        }
        uint32_t ent[GROUPS];
        uint32_t at[GROUPS];   // tile | rank << 12, or all ones
        // a turn within the segment needs no test of its steps (with that, and
        // the row of a bond from one product and no branch, 1000 runs of L =
        // 1024 take 14.0 ms, not 15.1; 3072 of L = 128 0.305, not 0.326)
        auto turn = [&](auto whole) __attribute__((always_inline)) {
            RecT *out = rec + t0;
#pragma unroll
            for (uint32_t i = 0; i < GROUPS; ++i) {
                const uint32_t t = t0 + i * 64u;
                const bool here = decltype(whole)::value || t < end;
                const bool ok = here && (uint32_t)e[i] < M;
                const TileBond b = tile_bond(g, ok ? e[i] : 0);
                const bool in = ok && !b.cross;
                const uint64_t peers = match_label(b.k, tile_bits, ballot(in));
                at[i] = 0xFFFFFFFFu;
                if (in) {
                    const uint32_t rank = lanes_below(peers);
                    const uint32_t before = my[b.k];
                    at[i] = b.k | ((before + rank) << 12);
                    if (rank == 0u)
                        my[b.k] = before + (uint32_t)__popcll(peers);
                }
                RecT ev = 0;
                if (ok && b.cross) {
                    const uint32_t hh = g.rows(b.tr);
                    const uint32_t iu = b.k * g.per + g.border(b.lr, b.lc, hh);
                    const uint32_t kv = b.down ? b.k + g.KW : b.k + 1u;
                    const uint32_t iv = kv * g.per + (b.down ? b.lc : g.border(b.lr, 0u, hh));
                    ev = EventBits<RecT>::join(iu, iv);
                }
                if (here)
                    out[i * 64u] = ev;
                ent[i] = TileEntry::make(t, b.lr * g.w + b.lc, b.down);
            }
        };
        if (base + 256u * GROUPS <= end)
            turn(std::true_type());
        else
            turn(std::false_type());
        t0 += 256u * GROUPS;
        load();
        __syncthreads();
        for (uint32_t k = tid; k < g.K; k += 256u) {
            uint32_t acc = cursor[k];
#pragma unroll
            for (uint32_t w = 0; w < 4u; ++w) {
                const uint32_t n = tile_dyn[w * g.K + k];
                tile_dyn[w * g.K + k] = acc;
                acc += n;
            }
            cursor[k] = acc;
            wrong |= acc > g.offset(k / g.KW, k % g.KW) + g.bonds_of(k);
        }
        if (__syncthreads_or(wrong))
            break;
#pragma unroll
        for (uint32_t i = 0; i < GROUPS; ++i)
            if (at[i] != 0xFFFFFFFFu)
                list[my[at[i] & 0xFFFu] + (at[i] >> 12)] = ent[i];
    }
    if (nseg == 1u) {
        for (uint32_t k = tid; k < g.K; k += 256u)
            wrong |= cursor[k] != g.offset(k / g.KW, k % g.KW) + g.bonds_of(k);
        const int any = __syncthreads_or(wrong);
        if (tid == 0u)
            odd[run] = any ? 1u : 0u;
    }
}

// One tile of one run on one wavefront: 64 of the tile's bonds at a time
// (lane = bond, in step order), as in sweep_run: finds, then rounds in which
// every candidate claims its roots and merges if it is the earliest claimant
// of each root it would change: of the closed one or ones, or, when both are
// open, of both.  No budget of rounds: the earliest pending candidate always merges.  Blocks of
// a run go to one XCD (shuf_block), whose L2 then collects the records that
// the run's tiles write into shared lines.
template <typename RecT>
__global__ __launch_bounds__(64) void tile_sweep_kernel(
    TileGeo g, uint32_t rn, const uint32_t *__restrict__ lists, int64_t list_stride,
    const uint32_t *__restrict__ windows, const uint16_t *__restrict__ init, RecT *__restrict__ records,
    int64_t rec_stride, uint32_t *__restrict__ span_step,
    const uint32_t *__restrict__ odd)
{
    extern __shared__ uint32_t tile_lds[];
    uint32_t *claims = tile_lds;
    uint32_t rl, k;
    if (!shuf_block(g.K, rn, rl, k) || odd[rl])
        return;
    const uint32_t lane = threadIdx.x;
    const uint32_t tr = k / g.KW, tc = k % g.KW;
    const uint32_t n = TileGeo::bonds(g.rows(tr), g.cols(tc));
    const uint32_t id0 = k * g.per - TILE_OPEN;   // an open code to its id
    const TileState st{(char *)(tile_lds + TILE_CLAIM_SLOTS)};
    const uint32_t below = 2u * g.w;   // from a node's code to the one below
    const uint32_t first = g.offset(tr, tc);
    const uint32_t *list = lists + (int64_t)rl * list_stride + first;
    RecT *rec_out = records + (int64_t)rl * rec_stride;
    {
        const uint4 *src = (const uint4 *)(init + (size_t)k * g.init_stride);
        uint4 *dst = (uint4 *)st.code;
        for (uint32_t i = lane; i < g.init_stride / 8u; i += 64u)
            dst[i] = src[i];
    }
    for (uint32_t i = lane; i < TILE_CLAIM_SLOTS; i += 64u)
        claims[i] = 0u;
    __syncthreads();

    // The window of the list's entries, and the entry the next one starts at.
    // (32-bit records: fewer steps than a window.)
    constexpr bool WINDOWS = sizeof(RecT) == 8u;
    const uint32_t M = 2u * g.L * (g.L - 1u);
    uint32_t window = 0;
    auto window_start = [&]() {
        const uint32_t w = window / TILE_WINDOW + 1u, W = tile_windows(M);
        return w < W ? windows[((size_t)rl * W + w) * g.K + k] - first : 0xFFFFFFFFu;
    };
    uint32_t next_window = WINDOWS ? window_start() : 0xFFFFFFFFu;

    // One batch: the bonds `cur` (entries at `at`), with the codes of the next batch's
    // endpoints (`next`) read before its merges (a parent read early is still
    // an ancestor).
    uint32_t hint_u = TILE_OPEN, hint_v = TILE_OPEN, tag = 0, span_at = PC_NO_SPAN;
    auto batch = [&](uint32_t at, uint32_t cur, uint32_t next, bool active) __attribute__((always_inline)) {
        uint32_t t, x, y, down;
        TileEntry::take(cur, t, x, down);
        if constexpr (WINDOWS) {
            t += window;
            while (next_window < at + 64u) {
                t += at + lane >= next_window ? TILE_WINDOW : 0u;
                window += TILE_WINDOW;
                next_window = window_start();
            }
        }
        y = x + (down ? below : 2u);
        x = st.is_root(hint_u) ? x : hint_u;
        y = st.is_root(hint_v) ? y : hint_v;
        uint32_t cx, cy;
        find2(st, x, cx, y, cy);
        {
            uint32_t tn, un, dn;
            TileEntry::take(next, tn, un, dn);
            hint_u = st.get(un);
            hint_v = st.get(un + (dn ? below : 2u));
        }
        bool cand = active && x != y;
        RecT rec = 0;
        while (ballot(cand)) {
            tag += 64u;
            const uint32_t mine = tag + 63u - lane;
            const bool open_x = cx < TILE_CLOSED, open_y = cy < TILE_CLOSED;
            // an open root is claimed only where two open ones may join: the
            // join waits for every earlier candidate of either root, which
            // else would name a root it was not yet joined with
            const bool join = open_x && open_y;
            const bool joins = ballot(cand && join) != 0u;
            const uint32_t su = (x >> 1) % TILE_CLAIM_SLOTS, sv = (y >> 1) % TILE_CLAIM_SLOTS;
            if (cand && (!open_x || joins))
                atomicMax(&claims[su], mine);
            if (cand && (!open_y || joins))
                atomicMax(&claims[sv], mine);
            const uint32_t held_x = claims[su], held_y = claims[sv];
            const bool go = cand && ((open_x && !join) || held_x == mine) &&
                            ((open_y && !join) || held_y == mine);
            // an open root is the parent of a closed one
            const uint32_t sx = cx & 0xFFFu, sy = cy & 0xFFFu;
            const bool x_big = open_x || (!open_y && sx >= sy);
            const bool closed = !open_x && !open_y;
            const uint32_t big = x_big ? x : y, small = x_big ? y : x;
            const uint32_t sides = (cx | cy) & 0x3000u;
            const bool spans_here = go && closed && sides == 0x3000u;
            if (go)
                st.set(small, big);
            if (go && closed)
                st.set(big, TILE_CLOSED + (spans_here ? 0u : sides) + sx + sy);
            if (go) {
                const uint32_t ix = id0 + cx, iy = id0 + cy;
                const uint32_t gain = ((open_x ? cy : cx) & 0x3FFFu) | EventBits<RecT>::top |
                                      (open_x ? 0u : 0x4000u);
                const uint32_t lo = join ? ix | EventBits<RecT>::top : open_x ? ix : iy;
                const uint32_t hi = join ? iy | EventBits<RecT>::top : gain;
                rec = pack_record<RecT>(closed ? sx : lo, closed ? sy : hi);
            }
            const uint64_t spans = ballot(spans_here);
            if (spans)
                span_at = min(span_at, read_lane(t, (uint32_t)__builtin_ctzll(spans)) + 1u);
            cand = cand && !go;
            if (!ballot(cand))
                break;
            if (cand)
                find2(st, x, cx, y, cy);
            cand = cand && x != y;
        }
        if (active && rec != 0)   // the others are 0 since tile_scatter
            rec_out[t] = rec;
    };
    // Entries are loaded two batches ahead, into registers that alternate: a
    // load in a branch, or one whose register is copied at the end of the
    // loop, would be waited for at once, with the stores before it.  Lanes
    // past the end read the last entry again.
    uint32_t e0 = list[min(lane, n - 1u)], e1 = list[min(64u + lane, n - 1u)];
    uint32_t base = 0;
    for (; base + 128u <= n; base += 128u) {
        const uint32_t a = e0;
        e0 = list[min(base + 128u + lane, n - 1u)];
        batch(base, a, e1, true);
        const uint32_t b = e1;
        e1 = list[min(base + 192u + lane, n - 1u)];
        batch(base + 64u, b, e0, true);
    }
    for (; base < n; base += 64u) {
        batch(base, e0, e1, base + lane < n);
        e0 = e1;
    }
    if (lane == 0u && span_at != PC_NO_SPAN)
        atomicMin(&span_step[rl], span_at);
}

// A run's open nodes with their codes in LDS (the HBM codes of GlobalState).
struct OpenLdsState {
    static constexpr bool LDS = true;
    uint32_t *code;
    __device__ __forceinline__ uint32_t get(uint32_t i) const { return code[i]; }
    __device__ __forceinline__ void set(uint32_t i, uint32_t v) const { code[i] = v; }
    __device__ __forceinline__ bool is_root(uint32_t v) const { return (v >> 31) != 0u; }
    __device__ __forceinline__ uint32_t root(uint32_t size, uint32_t f) const { return 0x80000000u | (f << 29) | size; }
    __device__ __forceinline__ void sync() const {}
    __device__ __forceinline__ void decode(uint32_t v, uint32_t &size, uint32_t &f) const
    {
        size = v & 0x1FFFFFFFu;
        f = (v >> 29) & 3u;
    }
};

// A run's events in step order, on one workgroup: EVENT_FINDERS wavefronts
// scan the records and find the events' roots, a window of
// EVENT_FINDERS * 64 * EVENT_SCAN steps ahead of the wavefront that merges
// them (the resolver), with one barrier per window.  Each finder takes a
// segment of the window's steps (loaded a window ahead), appends its events
// to its list in LDS and writes the roots found beside them; a find that
// runs beside the merges of the window before may stop at a root linked
// meanwhile, which is still an ancestor.  The resolver takes the events 64 at
// a time (lane = event; fewer than 64 wait for the next window) through the
// rounds of sweep_run: claims, independent merges and star merges into the
// hub (one wavefront for all of it: L = 1024, 1000 runs 25 ms, now 20; L =
// 256, 200 runs 0.67 ms, now 0.51).  A gain's closed cluster is a root of its own that no other event
// touches: it needs no claim and no store.
#define EVENT_SCAN 4u
#define EVENT_FINDERS 3u
#define EVENT_SEGMENT (64u * EVENT_SCAN)
#define EVENT_WINDOW (EVENT_FINDERS * EVENT_SEGMENT)
#define EVENT_GAIN 0x80000000u

// LDS: the claim table, then per event of two windows and of the waiting
// ones its step, its first root, and its second root or (EVENT_GAIN set) the
// closed cluster: order << 30 | sides << 28 | size; the lists' lengths.
struct EventLds {
    uint32_t claims[CLAIM_SLOTS];
    uint32_t t[2u * EVENT_WINDOW + 64u], a[2u * EVENT_WINDOW + 64u], b[2u * EVENT_WINDOW + 64u];
    uint32_t count[2u * EVENT_FINDERS + 2u];
};

template <class St, typename RecT>
__device__ __forceinline__ void event_run(const St &st, uint32_t M, RecT *rec_io,
                                          EventLds &ev, uint32_t *span_step)
{
    const uint32_t lane = threadIdx.x & 63u, wave = uniform(threadIdx.x >> 6);
    constexpr uint32_t TOP = EventBits<RecT>::top;
    uint32_t *const claims = ev.claims;
    const uint32_t windows = (M + EVENT_WINDOW - 1u) / EVENT_WINDOW;

    // a finder's window w: the segment's events into half w & 1 of the lists
    const uint32_t seg = wave ? (wave - 1u) * EVENT_SEGMENT : 0u;
    RecT ahead[EVENT_SCAN];
    auto load = [&](uint32_t w) {
#pragma unroll
        for (uint32_t i = 0; i < EVENT_SCAN; ++i)
            ahead[i] = rec_io[min(w * EVENT_WINDOW + seg + i * 64u + lane, M - 1u)];
    };
    auto find_window = [&](uint32_t w) {
        RecT cur[EVENT_SCAN];
#pragma unroll
        for (uint32_t i = 0; i < EVENT_SCAN; ++i)
            cur[i] = ahead[i];
        load(w + 1u);
        const uint32_t at = (w & 1u) * EVENT_WINDOW + seg, t0 = w * EVENT_WINDOW + seg;
        uint32_t n = 0;
#pragma unroll
        for (uint32_t i = 0; i < EVENT_SCAN; ++i) {
            const uint32_t t = t0 + i * 64u + lane;
            const bool is = EventBits<RecT>::is_event(cur[i]) && t < M;
            const uint64_t m = ballot(is);
            if (is) {
                uint32_t lo, hi;
                unpack_record(cur[i], lo, hi);
                const uint32_t p = at + n + lanes_below(m);
                ev.t[p] = t;
                ev.a[p] = lo & (TOP - 1u);
                ev.b[p] = (lo & TOP) ? hi & (TOP - 1u)
                                     : EVENT_GAIN | ((hi & 0x4000u) << 16) |
                                           ((hi & 0x3000u) << 16) | (hi & 0xFFFu);
            }
            n += (uint32_t)__popcll(m);
        }
        if (lane == 0u)
            ev.count[(w & 1u) * EVENT_FINDERS + wave - 1u] = n;
        for (uint32_t i = lane; i < n; i += 64u) {
            const uint32_t b = ev.b[at + i];
            uint32_t x = ev.a[at + i], y = (b & EVENT_GAIN) ? x : b, cx, cy;
            find2(st, x, cx, y, cy);
            ev.a[at + i] = x;
            if (!(b & EVENT_GAIN))
                ev.b[at + i] = y;
        }
    };

    uint32_t span_at = *span_step, tag = 0, waiting = 0;
    if (wave) {
        load(0u);
        find_window(0u);
    }
    __syncthreads();
    for (uint32_t w = 0; w < windows; ++w) {
        if (wave) {
            if (w + 1u < windows)
                find_window(w + 1u);
            st.sync();
            __syncthreads();
            continue;
        }
        uint32_t len[EVENT_FINDERS], total = waiting, done = 0;
#pragma unroll
        for (uint32_t f = 0; f < EVENT_FINDERS; ++f) {
            len[f] = uniform(ev.count[(w & 1u) * EVENT_FINDERS + f]);
            total += len[f];
        }
        // place of event i: the waiting ones, then the segments' lists
        auto place = [&](uint32_t i) {
            if (i < waiting)
                return 2u * EVENT_WINDOW + i;
            uint32_t j = i - waiting, p = (w & 1u) * EVENT_WINDOW;
#pragma unroll
            for (uint32_t f = 0; f + 1u < EVENT_FINDERS; ++f) {
                const bool past = j >= len[f];
                // the rest of the list, then the next segment
                p += past ? EVENT_SEGMENT : 0u;
                j -= past ? len[f] : 0u;
                if (!past)
                    break;
            }
            return p + j;
        };
        const bool last = w + 1u == windows;
        while (total - done >= 64u || (last && done < total)) {
        const uint32_t n = min(total - done, 64u);
        const bool active = lane < n;
        const uint32_t slot = place(done + min(lane, n - 1u));
        done += n;
        const uint32_t t = ev.t[slot], eb = ev.b[slot];
        const bool gain = active && (eb & EVENT_GAIN);
        const bool swap = gain && (eb & 0x40000000u);   // the closed cluster is on u's side
        uint32_t ru = ev.a[slot];
        uint32_t rv = (eb & EVENT_GAIN) ? ru : eb;
        uint32_t cu, cv;
        find2(st, ru, cu, rv, cv);
        if (gain) {
            rv = 0xFFFFFFFFu;
            cv = st.root(eb & 0xFFFu, (eb >> 28) & 3u);
        }
        bool cand = active && ru != rv;
        RecT rec = 0;
        while (ballot(cand)) {
            tag += 64u;
            const uint32_t mine = tag + 63u - lane;
            const uint32_t su = claim_slot(ru), sv = claim_slot(rv);
            if (cand)
                atomicMax(&claims[su], mine);
            if (cand && !gain)
                atomicMax(&claims[sv], mine);
            const uint32_t held_u = claims[su], held_v = gain ? mine : claims[sv];
            const bool own_u = held_u == mine, own_v = held_v == mine;
            bool go = cand && own_u && own_v;
            uint64_t star = 0;
            uint32_t hub = 0;
            const uint64_t blocked = ballot(cand && !go);
            if (blocked) {
                const uint32_t fl = (uint32_t)__builtin_ctzll(blocked);
                hub = read_lane(own_u ? rv : ru, fl);
                const bool at_u = ru == hub;
                const bool touch = cand && (at_u || rv == hub);
                const uint64_t tm = ballot(touch);
                const uint64_t bad = tm & ~ballot(touch && (at_u ? own_v : own_u));
                star = bad ? (tm & ((bad & (0u - bad)) - 1u)) : tm;
                go = go && !touch;
                const uint32_t hu = tag + 63u - held_u, hv = tag + 63u - held_v;
                const bool late = cand && !go && !((star >> lane) & 1u) &&
                                  (((star >> (hu & 63u)) & 1u) || ((star >> (hv & 63u)) & 1u));
                const uint64_t lm = ballot(late);
                if (lm)
                    star &= (lm & (0u - lm)) - 1u;
            }
            const bool in_star = (star >> lane) & 1u;
            if (star) {
                const bool at_u = ru == hub;
                const uint32_t x = at_u ? rv : ru;
                uint32_t sx, fx, sh, fh;
                st.decode(at_u ? cv : cu, sx, fx);
                st.decode(at_u ? cu : cv, sh, fh);
                const uint32_t first = (uint32_t)__builtin_ctzll(star);
                const uint32_t s_hub = read_lane(sh, first), f_hub = read_lane(fh, first);
                const uint32_t incl = wave_scan_add(in_star ? sx : 0u);
                const uint32_t total = read_lane(incl, 63u);
                const uint64_t m1 = ballot(in_star && (fx & 1u));
                const uint64_t m2 = ballot(in_star && (fx & 2u));
                const uint32_t f_all = f_hub | (m1 ? 1u : 0u) | (m2 ? 2u : 0u);
                if (in_star) {
                    if (!gain)
                        st.set(x, hub);
                    const uint32_t sh_now = s_hub + incl - sx;
                    rec = at_u != swap ? pack_record<RecT>(sh_now, sx) : pack_record<RecT>(sx, sh_now);
                }
                if (lane == first)
                    st.set(hub, st.root(s_hub + total, f_all == 3u ? 0u : f_all));
                if (f_all == 3u) {
                    const uint32_t l1 = (f_hub & 1u) ? first : (uint32_t)__builtin_ctzll(m1);
                    const uint32_t l2 = (f_hub & 2u) ? first : (uint32_t)__builtin_ctzll(m2);
                    span_at = min(span_at, read_lane(t, max(l1, l2)) + 1u);
                }
            }
            bool spans_here = false;
            if (go) {
                uint32_t sa, fa, sb, fb;
                st.decode(cu, sa, fa);
                st.decode(cv, sb, fb);
                const bool a_big = gain || sa >= sb;
                const uint32_t big = a_big ? ru : rv, small = a_big ? rv : ru;
                const uint32_t f = fa | fb;
                if (!gain)
                    st.set(small, big);
                st.set(big, st.root(sa + sb, f == 3u ? 0u : f));
                rec = swap ? pack_record<RecT>(sb, sa) : pack_record<RecT>(sa, sb);
                spans_here = f == 3u;
            }
            {
                const uint64_t spans = ballot(spans_here);
                if (spans)
                    span_at = min(span_at, read_lane(t, (uint32_t)__builtin_ctzll(spans)) + 1u);
            }
            cand = cand && !go && !in_star;
            st.sync();
            if (!ballot(cand))
                break;
            if (cand) {
                uint32_t z = gain ? ru : rv, cz = cv;
                find2(st, ru, cu, z, cz);
                if (!gain) {
                    rv = z;
                    cv = cz;
                }
            }
            cand = cand && ru != rv;
        }
        if (active)
            rec_io[t] = rec;
        }
        // fewer than a batch are left: they wait in front of the next window
        const uint32_t left = total - done;
        if (lane < left) {
            const uint32_t slot = place(done + lane);
            const uint32_t t = ev.t[slot], a = ev.a[slot], b = ev.b[slot];
            ev.t[2u * EVENT_WINDOW + lane] = t;
            ev.a[2u * EVENT_WINDOW + lane] = a;
            ev.b[2u * EVENT_WINDOW + lane] = b;
        }
        waiting = left;
        st.sync();
        __syncthreads();
    }
    if (threadIdx.x == 0u)
        *span_step = span_at;
}

// Codes in LDS (LDS_STATE) or in the run's slot of `states`; both start from
// `open` (tile_init_kernel).
template <typename RecT, bool LDS_STATE>
__global__ __launch_bounds__(64 * (1 + EVENT_FINDERS)) void event_sweep_kernel(
    uint32_t nodes, uint32_t M, const uint32_t *__restrict__ open,
    uint32_t *__restrict__ states, RecT *__restrict__ records, int64_t rec_stride,
    uint32_t *__restrict__ span_step, const uint32_t *__restrict__ odd)
{
    extern __shared__ uint32_t event_codes[];
    __shared__ EventLds ev;
    constexpr uint32_t T = 64u * (1u + EVENT_FINDERS);
    if (odd[blockIdx.x])
        return;
    RecT *rec = records + (int64_t)blockIdx.x * rec_stride;
    uint32_t *code = LDS_STATE ? event_codes : states + (size_t)blockIdx.x * nodes;
    for (uint32_t i = threadIdx.x; i < CLAIM_SLOTS; i += T)
        ev.claims[i] = 0u;
    for (uint32_t i = threadIdx.x; i < nodes; i += T)
        code[i] = open[i];
    __threadfence_block();
    __syncthreads();
    if constexpr (LDS_STATE)
        event_run<OpenLdsState, RecT>(OpenLdsState{code}, M, rec, ev, span_step + blockIdx.x);
    else
        event_run<GlobalState, RecT>(GlobalState{code}, M, rec, ev, span_step + blockIdx.x);
}

// Running per-run state (after some number of bonds).
template <bool WIDE>
struct RunState {
    using MT = typename Wide<WIDE>::T;
    uint64_t mx, merges, s2;
    MT s3, s4;
};

template <bool WIDE>
__device__ __forceinline__ RunState<WIDE> load_state(const uint64_t *cs)
{
    RunState<WIDE> st;
    st.mx = cs[0];
    st.merges = cs[1];
    st.s2 = cs[2];
    if constexpr (WIDE) {
        st.s3 = (u128)cs[3] | ((u128)cs[4] << 64);
        st.s4 = (u128)cs[5] | ((u128)cs[6] << 64);
    } else {
        st.s3 = cs[3];
        st.s4 = cs[5];
    }
    return st;
}

// State after each lane's step: chunk-start state plus the inclusive scan
// of the deltas of the chunk's records.
template <bool WIDE>
__device__ __forceinline__ RunState<WIDE> advance(const RunState<WIDE> &st0,
                                                  Deltas<WIDE> d)
{
    RunState<WIDE> st;
    st.merges = st0.merges + scan_count(d.merge());
    scan_state(d.dmax, d.d2, d.d3, d.d4);
    st.mx = umax64(st0.mx, (uint64_t)d.dmax);
    st.s2 = st0.s2 + d.d2;
    st.s3 = st0.s3 + d.d3;
    st.s4 = st0.s4 + d.d4;
    return st;
}

// The seven observables from a state: x[0] max, x[1] spanning, x[2..6]
// moments k = 0..4 of all clusters but one largest.
template <bool WIDE>
__device__ __forceinline__ void observables(const RunState<WIDE> &st,
                                            uint32_t N, bool span,
                                            typename Wide<WIDE>::T x[7])
{
    using MT = typename Wide<WIDE>::T;
    const uint64_t m = st.mx;
    x[0] = (MT)m;
    x[1] = (MT)(span ? 1u : 0u);
    x[2] = (MT)((uint64_t)N - st.merges - 1u);
    x[3] = (MT)((uint64_t)N - m);
    const MT m2 = (MT)(m * m);
    x[4] = (MT)st.s2 - m2;
    x[5] = st.s3 - m2 * (MT)m;
    x[6] = st.s4 - m2 * m2;
}

// ---------------------------------------------------------------------------
// chunk_scan in two passes.  (A) chunk_delta: every (run, chunk) in
// parallel, the totals of the chunk's deltas {max merged size, merges, dS2,
// dS3, dS4} reduced across the wave into that chunk's entry.  (B)
// chunk_prefix: one wavefront per run turns the entries in place into the
// state at the start of each chunk, 64 chunks per step (scans across lanes,
// a carry between steps).
// ---------------------------------------------------------------------------
#define CHUNK_DELTA_PER_BLOCK 8u

template <typename RecT, bool WIDE>
__global__ __launch_bounds__(64) void chunk_delta_kernel(
    uint32_t M, const RecT *__restrict__ records, int64_t rec_stride,
    uint64_t *__restrict__ chunk_state)
{
    // blocks: run-major, CHUNK_DELTA_PER_BLOCK chunks each
    const uint32_t C = (M + 63u) / 64u;
    const uint32_t per_run = (C + CHUNK_DELTA_PER_BLOCK - 1u) / CHUNK_DELTA_PER_BLOCK;
    const uint32_t r = blockIdx.x / per_run, lane = threadIdx.x;
    const RecT *rec_r = records + (int64_t)r * rec_stride;
    uint64_t *out = chunk_state + (size_t)r * C * PC_STATE_WORDS;
    const uint32_t c0 = (blockIdx.x % per_run) * CHUNK_DELTA_PER_BLOCK + lane / 16u;
    // a row of 16 lanes per chunk, four records a lane (their order within a
    // chunk does not matter to its totals): a quarter of the scan steps of a
    // lane per record, and four of six levels.  With the scans in place, 10^4
    // runs of L = 128 take 0.33 ms (1.35 before), 1000 of L = 1024 3.4 (10.8)
    constexpr uint32_t ITER = CHUNK_DELTA_PER_BLOCK / 4u;
    RecT rec[ITER][4];
#pragma unroll
    for (uint32_t i = 0; i < ITER; ++i)
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u) {
            const uint32_t q = (c0 + 4u * i) * 64u + u * 16u + lane % 16u;
            rec[i][u] = rec_r[min(q, M - 1u)];
            if (q >= M)
                rec[i][u] = 0;
        }
#pragma unroll
    for (uint32_t i = 0; i < ITER; ++i) {
        const uint32_t c = c0 + 4u * i;
        Deltas<WIDE> d(rec[i][0]);
        uint32_t cnt = (uint32_t)__popcll(ballot(d.merge()) >> (lane & 48u) & 0xFFFFull);
#pragma unroll
        for (uint32_t u = 1; u < 4u; ++u) {
            const Deltas<WIDE> e(rec[i][u]);
            cnt += (uint32_t)__popcll(ballot(e.merge()) >> (lane & 48u) & 0xFFFFull);
            d.dmax = max(d.dmax, e.dmax);
            d.d2 += e.d2;
            d.d3 += e.d3;
            d.d4 += e.d4;
        }
        scan_state_rows(d.dmax, d.d2, d.d3, d.d4);
        if (lane % 16u == 15u && c < C) {
            const uint64_t hi3 = WIDE ? (uint64_t)((u128)d.d3 >> 64) : 0u;
            const uint64_t hi4 = WIDE ? (uint64_t)((u128)d.d4 >> 64) : 0u;
            uint64_t *w = out + (size_t)c * PC_STATE_WORDS;
            w[0] = d.dmax;
            w[1] = cnt;
            w[2] = d.d2;
            w[3] = (uint64_t)d.d3;
            w[4] = hi3;
            w[5] = (uint64_t)d.d4;
            w[6] = hi4;
            w[7] = 0u;
        }
    }
}

template <bool WIDE>
__global__ __launch_bounds__(64) void chunk_prefix_kernel(
    uint32_t N, uint32_t M, uint64_t *__restrict__ chunk_state)
{
    using MT = typename Wide<WIDE>::T;
    const uint32_t r = blockIdx.x, lane = threadIdx.x;
    const uint32_t C = (M + 63u) / 64u;
    uint64_t *st = chunk_state + (size_t)r * C * PC_STATE_WORDS;
    // state at the start of the current group of 64 chunks
    uint64_t mx = 1, merges = 0, s2 = N;
    MT s3 = N, s4 = N;
    for (uint32_t c0 = 0; c0 < C; c0 += 64u) {
        const uint32_t c = c0 + lane;
        uint64_t w[PC_STATE_WORDS] = {0, 0, 0, 0, 0, 0, 0, 0};
        if (c < C)
            for (uint32_t k = 0; k < PC_STATE_WORDS; ++k)
                w[k] = st[(size_t)c * PC_STATE_WORDS + k];
        const uint32_t dmax = (uint32_t)w[0];
        const uint64_t cnt = w[1], d2 = w[2];
        MT d3 = (MT)w[3], d4 = (MT)w[5];
        if constexpr (WIDE) {
            d3 |= (MT)w[4] << 64;
            d4 |= (MT)w[6] << 64;
        }
        uint32_t imax = dmax;
        const uint32_t icnt = wave_scan_add((uint32_t)cnt);
        typename Deltas<WIDE>::D2 id2 = (typename Deltas<WIDE>::D2)d2;
        MT id3 = d3, id4 = d4;
        scan_state(imax, id2, id3, id4);
        // exclusive prefix: the sums minus the own chunk, the maximum of the
        // chunks before (the previous lane's inclusive maximum)
        uint32_t emax = (uint32_t)__shfl_up((int)imax, 1, 64);
        if (lane == 0)
            emax = 0u;
        if (c < C)
            for (uint32_t k = 0; k < PC_STATE_WORDS; ++k)
                st[(size_t)c * PC_STATE_WORDS + k] = state_word(
                    k, umax64(mx, emax), merges + icnt - cnt, s2 + id2 - d2,
                    s3 + id3 - d3, s4 + id4 - d4);
        mx = umax64(mx, read_lane(imax, 63u));
        merges += read_lane(icnt, 63u);
        s2 += read_lane(id2, 63u);
        s3 += read_lane(id3, 63u);
        s4 += read_lane(id4, 63u);
    }
}

// ---------------------------------------------------------------------------
// Microcanonical sums: block (chunk c, run group g), lane = step.  Each lane
// accumulates its step's sums over its wave's runs of the group in registers;
// the waves add up in LDS, groups combine through multi-word atomics.
// ---------------------------------------------------------------------------
// Workgroups of one wave fill the GPU where there are 8192 of them with 32
// runs each; they use no LDS, which the sweeps beside them hold (10^4 runs of
// L = 128 as a pipeline: 8.3 ms, 9.5 with the form below).  Elsewhere the four
// waves of a workgroup share 64 runs of a chunk and add up in LDS, so that a
// fourth of the atomics remain (L = 100, 500 runs 0.121 -> 0.044 ms; L = 16,
// 40 runs 13 -> 8 us).  Bound by vector issue.  With the squares added up limb
// by limb (SquareSum) instead of as 128- and 192-bit integers, and the sums of
// N - max left to the end, 1000 runs of L = 1024 take 9.3 ms, not 12.7 (their
// records alone: 3.5); 600 of L = 181 0.196, not 0.262; 200 of L = 256 0.147,
// not 0.180; a sub-batch of L = 128 beside its sweeps 0.17, not 0.21.
#define SUMS_BLOCKS 8192u
#define SUMS_RUNS 32u
// Few runs added to sums that are there take a wave each, as long as their
// atomics cost less than the waves' way through LDS: up to SUMS_FEW chunks of
// all runs, SUMS_FEW_ONE of one (16 runs of L = 16 12.6 us a call, so 11.7; 2
// of L = 64 11.2 and 11.3, 8 of them 12.0 and 16.9; one of L = 128 12.6 and
// 11.7, of L = 512 100 and 103).
#define SUMS_FEW 192u
#define SUMS_FEW_ONE 4096u
#define SUMS_MOST 1024u   // runs a group may hold: what the bounds below allow

// Product of two numbers below 2^24 (two full-rate instructions; __umul24
// returns an int).
__device__ __forceinline__ uint64_t mul24_wide(uint32_t a, uint32_t b)
{
    uint32_t hi;
    asm("v_mul_hi_u32_u24 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
    return ((uint64_t)hi << 32) | (uint32_t)__umul24(a, b);
}

// Product of numbers below 2^44 and 2^44 (the high words' below 2^24).
__device__ __forceinline__ u96 mul_u96(uint64_t p, uint64_t q)
{
    const uint32_t pl = (uint32_t)p, ph = (uint32_t)(p >> 32), ql = (uint32_t)q,
                   qh = (uint32_t)(q >> 32);
    const uint64_t t0 = (uint64_t)pl * ql, t1 = (uint64_t)pl * qh + (t0 >> 32),
                   t2 = (uint64_t)ph * ql + (uint32_t)t1;
    const uint32_t hi = (uint32_t)__umul24(ph, qh) + (uint32_t)(t1 >> 32) + (uint32_t)(t2 >> 32);
    return ((u96)hi << 64) | ((u96)(uint32_t)t2 << 32) | (uint32_t)t0;
}

// Sum of the squares of numbers of K limbs of B <= 27 bits: a sum for every
// product of two limbs, put together once at the end, so that a square costs
// no carries.  SUMS_MOST products below 2^54 fit 64 bits, and a product is
// added by the instruction that forms it (in doubles, limbs of 21 bits and a
// conversion each, 1000 runs of L = 1024 took 10.3 ms, with these 9.3).
template <int K, int B>
struct SquareSum {
    static_assert(2 * B <= 54, "64 bits hold the sums");
    uint64_t sum[K * (K + 1) / 2] = {};
    __device__ __forceinline__ void add(const uint32_t *limb)
    {
        int n = 0;
#pragma unroll
        for (int i = 0; i < K; ++i)
#pragma unroll
            for (int j = i; j < K; ++j)
                sum[n] += (uint64_t)limb[i] * limb[j], ++n;
    }
    // low 128 bits, and the word above
    __device__ __forceinline__ u128 value(uint64_t &top) const
    {
        u128 lo = 0;
        top = 0;
        int n = 0;
#pragma unroll
        for (int i = 0; i < K; ++i)
#pragma unroll
            for (int j = i; j < K; ++j) {
                const u128 v = (u128)sum[n++] << (i == j ? 0 : 1);
                const int shift = B * (i + j);
                const u128 part = shift < 128 ? v << (shift & 127) : (u128)0;
                lo += part;
                top += lo < part ? 1u : 0u;
                top += shift >= 128 ? (uint64_t)(v << (shift & 127))
                                    : shift ? (uint64_t)(v >> ((128 - shift) & 127)) : 0u;
            }
        return lo;
    }
};

template <typename RecT, bool WIDE, uint32_t WAVES>
__global__ __launch_bounds__(64 * WAVES) void micro_sums_kernel(
    uint32_t N, uint32_t M, uint32_t R, uint32_t runs_per_group,
    const RecT *__restrict__ records, int64_t rec_stride,
    const uint32_t *__restrict__ span_step,
    const uint64_t *__restrict__ chunk_state, uint64_t *__restrict__ sum1,
    uint64_t *__restrict__ sum2, bool store)
{
    // the waves' accumulators on their way to wave 0
    constexpr uint32_t PARTS = WIDE ? 21u : 18u;
    __shared__ uint64_t part[WAVES > 1u ? PARTS : 1u][64];
    const uint32_t c = blockIdx.x, g = blockIdx.y, lane = threadIdx.x & 63u;
    const uint32_t wave = uniform(threadIdx.x >> 6);
    const uint32_t C = (M + 63u) / 64u;
    const uint64_t S = (uint64_t)M + 1u;
    const uint32_t q = c * 64u + lane, s = q + 1u;
    const bool valid = q < M;
    const uint32_t r0 = g * runs_per_group;
    const uint32_t r1 = min(R, r0 + runs_per_group);

    // the next run's state, record and spanning step, loaded a run ahead
    RunState<WIDE> st_next;
    RecT rec_next;
    uint32_t span_next;
    auto ahead = [&](uint32_t r) __attribute__((always_inline)) {
        st_next = load_state<WIDE>(chunk_state + ((size_t)r * C + c) * PC_STATE_WORDS);
        rec_next = records[(int64_t)r * rec_stride + min(q, M - 1u)];
        span_next = span_step[r];
    };
    ahead(min(r0 + wave, R - 1u));

    // wave 3's sums to wave 2, whose sum goes to wave 1, and on to wave 0
    auto to_wave0 = [&](auto &&each) {
        if constexpr (WAVES > 1u)
        for (int w = WAVES - 1; w >= 0; --w) {
            if ((int)wave == w) {
                if (w + 1 < (int)WAVES)
                    each([&](uint32_t i, auto &v) {
                        using V = std::remove_reference_t<decltype(v)>;
                        if constexpr (sizeof(V) == 16)
                            v += (u128)part[i][lane] | ((u128)part[i + 1u][lane] << 64);
                        else
                            v += (V)part[i][lane];
                    });
                if (w > 0)
                    each([&](uint32_t i, auto &v) {
                        part[i][lane] = (uint64_t)v;
                        if constexpr (sizeof(v) == 16)
                            part[i + 1u][lane] = (uint64_t)(v >> 64);
                    });
            }
            __syncthreads();
        }
    };

    u128 acc1[7];
    u128 acc2[7];
    uint64_t acc2_top[7];
#pragma unroll
    for (int k = 0; k < 7; ++k) {
        acc1[k] = 0;
        acc2[k] = 0;
        acc2_top[k] = 0;
    }

    if constexpr (!WIDE) {
        // N <= 2^14 and at most SUMS_MOST runs per group bound every
        // accumulator: max, #clusters - 1 and N - max are below 2^14 (group
        // sums of squares below 2^38); the spanning flag is 0 or 1; moment 2
        // is below N^2 / 2 (squares below 2^54), moment 3 below N^3 / 4 =
        // 2^40, moment 4 below N^4 / 8 = 2^53.  The sums of N - max follow
        // from those of max.
        uint32_t n1[4] = {0, 0, 0, 0};  // sum x: max, span, #clusters - 1, N - max
        uint64_t n2[4] = {0, 0, 0, 0};  // sum x^2 of the same
        uint64_t m1_2 = 0, m1_3 = 0, m1_4 = 0;   // sum x: moments 2 to 4
        uint64_t sq_2 = 0;
        SquareSum<2, 27> sq_3, sq_4;
        uint32_t count = 0;
        for (uint32_t r = r0 + wave; r < r1; r += WAVES) {
            const RunState<false> st0 = st_next;
            const RecT rec = valid ? rec_next : (RecT)0;
            const uint32_t span = span_next;
            ahead(min(r + WAVES, r1 - 1u));
            ++count;
            Deltas<false> d(rec);
            const uint32_t merges = (uint32_t)st0.merges + scan_count(d.merge());
            scan_state(d.dmax, d.d2, d.d3, d.d4);
            const uint32_t mx = max((uint32_t)st0.mx, d.dmax), mx2 = (uint32_t)__umul24(mx, mx);
            const uint32_t x2 = N - merges - 1u;
            n1[0] += mx;
            n2[0] += mx2;
            n1[1] += s >= span ? 1u : 0u;
            n1[2] += x2;
            n2[2] += (uint32_t)__umul24(x2, x2);
            const uint32_t x4 = (uint32_t)st0.s2 + d.d2 - mx2;
            m1_2 += x4;
            sq_2 += (uint64_t)x4 * x4;
            const uint64_t x5 = st0.s3 + d.d3 - (uint64_t)mx2 * mx;
            m1_3 += x5;
            const uint64_t x6 = st0.s4 + d.d4 - (uint64_t)mx2 * mx2;
            m1_4 += x6;
            constexpr uint32_t LIMB = (1u << 27) - 1u;
            const uint32_t l5[2] = {(uint32_t)x5 & LIMB, (uint32_t)(x5 >> 27)};
            const uint32_t l6[2] = {(uint32_t)x6 & LIMB, (uint32_t)(x6 >> 27)};
            sq_3.add(l5);
            sq_4.add(l6);
        }
        n2[1] = n1[1];
        n1[3] = count * N - n1[0];
        n2[3] = (uint64_t)count * N * N + n2[0] - 2ull * N * n1[0];
        uint64_t none;
        u128 m2_2 = sq_2, m2_3 = sq_3.value(none), m2_4 = sq_4.value(none);
        to_wave0([&](auto &&at) {
#pragma unroll
            for (uint32_t k = 0; k < 4u; ++k) {
                at(k, n1[k]);
                at(4u + k, n2[k]);
            }
            at(8u, m1_2);
            at(9u, m1_3);
            at(10u, m1_4);
            at(12u, m2_2);
            at(14u, m2_3);
            at(16u, m2_4);
        });
        // column order of the sums: max, span, moments 0..4
        const int col[4] = {0, 1, 2, 3};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            acc1[col[k]] = n1[k];
            acc2[col[k]] = n2[k];
        }
        acc1[4] = m1_2;
        acc2[4] = m2_2;
        acc1[5] = m1_3;
        acc2[5] = m2_3;
        acc1[6] = m1_4;
        acc2[6] = m2_4;
    } else {
        // N <= 2^21 (the sums' limit) and at most SUMS_MOST runs per group:
        // S3 is below N^3 <= 2^63 (its deltas and scan stay in 64 bits), S4
        // at most N^4 <= 2^84 (96 bits); max, #clusters - 1 and N - max are
        // at most 2^21 (group sums below 2^32, of squares below 2^53),
        // moment 2 below 2^42, moment 3 below 2^63 and moment 4 below 2^84.
        // The sums of N - max follow from those of max.
        uint64_t n1[5] = {0, 0, 0, 0, 0}; // sum x: max, span, #clusters - 1, N - max, moment 2
        uint64_t n2[4] = {0, 0, 0, 0};    // sum x^2 of the first four
        uint32_t s_mx = 0, s_span = 0, s_cl = 0, count = 0;
        u96 s_3 = 0, s_4 = 0;             // sum x: moments 3 and 4
        // 32-bit records: N <= 2^16, moments below 2^31, 2^48 and 2^64
        constexpr int K3 = sizeof(RecT) == 4u ? 2 : 3, K4 = sizeof(RecT) == 4u ? 3 : 4;
        SquareSum<2, 27> sq_2;
        SquareSum<K3, 27> sq_3;
        SquareSum<K4, 27> sq_4;
        constexpr uint32_t LIMB = (1u << 27) - 1u;
        for (uint32_t r = r0 + wave; r < r1; r += WAVES) {
            const uint32_t mx0 = (uint32_t)st_next.mx, merges0 = (uint32_t)st_next.merges;
            const uint64_t s2_0 = st_next.s2, s3_0 = (uint64_t)st_next.s3;
            const u96 s4_0 = (u96)st_next.s4;
            const RecT rec = valid ? rec_next : (RecT)0;
            const uint32_t span = span_next;
            ahead(min(r + WAVES, r1 - 1u));
            ++count;
            uint32_t a, b;
            unpack_record(rec, a, b);
            // sizes below 2^21 + 1: 24-bit products, q <= 2^40
            uint32_t mxd = a + b;
            const uint32_t sz = mxd;
            const uint64_t qq = mul24_wide(a, b);
            uint64_t d2 = 2u * qq;
            uint64_t d3 = (uint64_t)(uint32_t)qq * (3u * sz) +
                          ((uint64_t)(uint32_t)__umul24((uint32_t)(qq >> 32), 3u * sz) << 32);
            u96 d4 = mul_u96(2u * qq, 2u * mul24_wide(sz, sz) - qq);
            const uint32_t merges = merges0 + scan_count(rec != 0);
            scan_state(mxd, d2, d3, d4);
            const uint32_t mx = max(mx0, mxd), cl = N - merges - 1u;
            const uint64_t m2 = mul24_wide(mx, mx);
            s_mx += mx;
            n2[0] += m2;
            s_span += s >= span ? 1u : 0u;
            s_cl += cl;
            n2[2] += mul24_wide(cl, cl);
            const uint64_t x4 = s2_0 + d2 - m2;
            const uint64_t x5 = s3_0 + d3 - ((uint64_t)(uint32_t)m2 * mx +
                                             ((uint64_t)(uint32_t)__umul24((uint32_t)(m2 >> 32), mx) << 32));
            const u96 x6 = s4_0 + d4 - mul_u96(m2, m2);
            n1[4] += x4;
            s_3 += x5;
            s_4 += x6;
            const uint32_t l4[2] = {(uint32_t)x4 & LIMB, (uint32_t)(x4 >> 27)};
            uint32_t l5[K3], l6[K4];
#pragma unroll
            for (int i = 0; i < K3; ++i)
                l5[i] = (uint32_t)(x5 >> (27 * i)) & (i + 1 < K3 ? LIMB : 0xFFFFFFFFu);
#pragma unroll
            for (int i = 0; i < K4; ++i)
                l6[i] = (uint32_t)(x6 >> (27 * i)) & (i + 1 < K4 ? LIMB : 0xFFFFFFFFu);
            sq_2.add(l4);
            sq_3.add(l5);
            sq_4.add(l6);
        }
        n1[0] = s_mx;
        n1[1] = n2[1] = s_span;
        n1[2] = s_cl;
        n1[3] = (uint64_t)count * N - s_mx;
        n2[3] = (uint64_t)count * N * N + n2[0] - 2ull * N * s_mx;
        uint64_t none, t2_3, t2_4;
        u128 m2_2 = sq_2.value(none), m2_3 = sq_3.value(t2_3), m2_4 = sq_4.value(t2_4);
        u128 m1_3 = s_3, m1_4 = s_4;
        {
            // the carries of the two 192-bit sums go with their low words
            u128 *const low[2] = {&m2_3, &m2_4};
            uint64_t *const top[2] = {&t2_3, &t2_4};
            to_wave0([&](auto &&at) {
#pragma unroll
                for (uint32_t k = 0; k < 5u; ++k)
                    at(k, n1[k]);
#pragma unroll
                for (uint32_t k = 0; k < 4u; ++k)
                    at(5u + k, n2[k]);
                at(9u, m2_2);
                at(11u, m1_3);
                at(13u, m1_4);
#pragma unroll
                for (uint32_t k = 0; k < 2u; ++k) {
                    const u128 before = *low[k];
                    at(15u + 3u * k, *low[k]);
                    *top[k] += *low[k] < before ? 1u : 0u;
                    at(17u + 3u * k, *top[k]);
                }
            });
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            acc1[k] = n1[k];
            acc2[k] = n2[k];
        }
        acc1[4] = n1[4];
        acc2[4] = m2_2;
        acc1[5] = m1_3;
        acc2[5] = m2_3;
        acc2_top[5] = t2_3;
        acc1[6] = m1_4;
        acc2[6] = m2_4;
        acc2_top[6] = t2_4;
    }

    if (wave)
        return;
    if (store && valid) {
#pragma unroll
        for (int k = 0; k < 7; ++k) {
            uint64_t *w1 = sum1 + ((uint64_t)k * S + s) * 2u, *w2 = sum2 + ((uint64_t)k * S + s) * 3u;
            w1[0] = (uint64_t)acc1[k];
            w1[1] = (uint64_t)(acc1[k] >> 64);
            w2[0] = (uint64_t)acc2[k];
            w2[1] = (uint64_t)(acc2[k] >> 64);
            w2[2] = acc2_top[k];
        }
    } else if (valid) {
#pragma unroll
        for (int k = 0; k < 7; ++k) {
            atomic_add_u128(sum1 + ((uint64_t)k * S + s) * 2u, acc1[k]);
            atomic_add_u192(sum2 + ((uint64_t)k * S + s) * 3u,
                            (uint64_t)acc2[k], (uint64_t)(acc2[k] >> 64),
                            acc2_top[k]);
        }
    }
    if (c == 0 && lane == 0 && r1 > r0) {
        // step 0: max 1, no spanning, every moment N - 1
        const u128 n = r1 - r0;
        const u128 x0[7] = {1, 0, N - 1u, N - 1u, N - 1u, N - 1u, N - 1u};
        for (int k = 0; k < 7; ++k) {
            const u128 sq = n * x0[k] * x0[k];
            if (store) {
                uint64_t *w1 = sum1 + (uint64_t)k * S * 2u, *w2 = sum2 + (uint64_t)k * S * 3u;
                w1[0] = (uint64_t)(n * x0[k]);
                w1[1] = (uint64_t)(n * x0[k] >> 64);
                w2[0] = (uint64_t)sq;
                w2[1] = (uint64_t)(sq >> 64);
                w2[2] = 0u;
                continue;
            }
            atomic_add_u128(sum1 + (uint64_t)k * S * 2u, n * x0[k]);
            atomic_add_u192(sum2 + (uint64_t)k * S * 3u, (uint64_t)sq,
                            (uint64_t)(sq >> 64), 0u);
        }
    }
}

// Step 0 alone (graphs without edges): max 1, no spanning, moments N - 1.
__global__ void step0_sums_kernel(uint32_t N, uint32_t R, uint64_t S,
                                  uint64_t *__restrict__ sum1,
                                  uint64_t *__restrict__ sum2)
{
    const u128 n = R;
    const u128 x0[7] = {1, 0, N - 1u, N - 1u, N - 1u, N - 1u, N - 1u};
    for (int k = 0; k < 7; ++k) {
        atomic_add_u128(sum1 + (uint64_t)k * S * 2u, n * x0[k]);
        const u128 sq = n * x0[k] * x0[k];
        atomic_add_u192(sum2 + (uint64_t)k * S * 3u, (uint64_t)sq,
                        (uint64_t)(sq >> 64), 0u);
    }
}

__global__ void expand_step0_kernel(uint32_t N, uint32_t R, uint64_t S,
                                    uint32_t *__restrict__ out_max,
                                    uint8_t *__restrict__ out_span,
                                    uint64_t *__restrict__ out_mom)
{
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= R)
        return;
    const uint64_t row = (uint64_t)r * S;
    out_max[row] = 1u;
    out_span[row] = 0u;
    for (int k = 0; k < 5; ++k)
        out_mom[row * 5u + k] = (uint64_t)N - 1u;
}

__global__ void fill_zero_kernel(uint64_t *__restrict__ p, uint64_t n)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = 0;
}

// ---------------------------------------------------------------------------
// Per-run traces: block (chunk c, run r), lane = step.
// ---------------------------------------------------------------------------
template <typename RecT, bool WIDE>
__global__ __launch_bounds__(64) void expand_kernel(
    uint32_t N, uint32_t M, const RecT *__restrict__ records,
    int64_t rec_stride, const uint32_t *__restrict__ span_step,
    const uint64_t *__restrict__ chunk_state, uint32_t *__restrict__ out_max,
    uint8_t *__restrict__ out_span, uint64_t *__restrict__ out_mom)
{
    using MT = typename Wide<WIDE>::T;
    const uint32_t c = blockIdx.x, r = blockIdx.y, lane = threadIdx.x;
    const uint32_t C = (M + 63u) / 64u;
    const uint64_t S = (uint64_t)M + 1u;
    const uint32_t q = c * 64u + lane, s = q + 1u;
    const bool valid = q < M;
    const RunState<WIDE> st0 = load_state<WIDE>(
        chunk_state + ((size_t)r * C + c) * PC_STATE_WORDS);
    const RecT rec = valid ? records[(int64_t)r * rec_stride + q] : (RecT)0;
    const RunState<WIDE> st = advance<WIDE>(st0, Deltas<WIDE>(rec));
    MT x[7];
    observables<WIDE>(st, N, s >= span_step[r], x);
    const uint64_t row = (uint64_t)r * S + s;
    if (valid) {
        out_max[row] = (uint32_t)x[0];
        out_span[row] = (uint8_t)x[1];
    }
    // the chunk's moments through LDS, so that a store takes 512 bytes in a row
    // (500 runs of L = 100: 97 us, with 64 pieces of 8 a store 122; a copy
    // writes their 445 MB in 91)
    __shared__ uint64_t mom[64 * 5];
#pragma unroll
    for (int k = 0; k < 5; ++k)
        mom[lane * 5u + k] = (uint64_t)x[2 + k];
    __syncthreads();
    const uint32_t n = min(64u, M - c * 64u) * 5u;
    uint64_t *dst = out_mom + ((uint64_t)r * S + c * 64u + 1u) * 5u;
#pragma unroll
    for (uint32_t i = 0; i < 5u; ++i)
        if (i * 64u + lane < n)
            dst[i * 64u + lane] = mom[i * 64u + lane];
    if (c == 0 && lane == 0) {
        const uint64_t row0 = (uint64_t)r * S;
        out_max[row0] = 1u;
        out_span[row0] = 0u;
        for (int k = 0; k < 5; ++k)
            out_mom[row0 * 5u + k] = (uint64_t)N - 1u;
    }
}


// The same as rows of the reference's structured array, packed: step (u32),
// edge (u32), spanning (one byte, with SPAN), largest cluster (u32), moments
// (5 u64).  A chunk's rows are laid out in LDS and go out as aligned words.
// One copy to the host then takes the place of one per field and of putting
// the fields together there: 40 runs of 32 x 32 nodes, 1.44 -> 1.00 ms a call.
template <typename RecT, bool WIDE, bool SPAN>
__global__ __launch_bounds__(64) void expand_rows_kernel(
    uint32_t N, uint32_t M, const int32_t *__restrict__ perm, int64_t perm_stride,
    const RecT *__restrict__ records, int64_t rec_stride,
    const uint32_t *__restrict__ span_step, const uint64_t *__restrict__ chunk_state,
    uint8_t *__restrict__ out)
{
    using MT = typename Wide<WIDE>::T;
    constexpr uint32_t ROW = SPAN ? 53u : 52u;
    __shared__ uint8_t rows[65u * ROW];
    const uint32_t c = blockIdx.x, r = blockIdx.y, lane = threadIdx.x;
    const uint32_t C = (M + 63u) / 64u;
    const uint64_t S = (uint64_t)M + 1u;
    const uint32_t q = c * 64u + lane, s = q + 1u;
    const bool valid = q < M;
    const RunState<WIDE> st0 = load_state<WIDE>(
        chunk_state + ((size_t)r * C + c) * PC_STATE_WORDS);
    const RecT rec = valid ? records[(int64_t)r * rec_stride + q] : (RecT)0;
    const uint32_t edge = valid ? (uint32_t)perm[(int64_t)r * perm_stride + q] : 0u;
    const RunState<WIDE> st = advance<WIDE>(st0, Deltas<WIDE>(rec));
    MT x[7];
    observables<WIDE>(st, N, s >= span_step[r], x);
    auto put = [&](uint32_t at, uint32_t step, uint32_t e, const MT *v) {
        uint8_t *w = rows + at * ROW;
        const uint32_t mx = (uint32_t)v[0];
        __builtin_memcpy(w, &step, 4);
        __builtin_memcpy(w + 4, &e, 4);
        if (SPAN)
            w[8] = (uint8_t)v[1];
        __builtin_memcpy(w + ROW - 44u, &mx, 4);
        for (int k = 0; k < 5; ++k) {
            const uint64_t m = (uint64_t)v[2 + k];
            __builtin_memcpy(w + ROW - 40u + 8 * k, &m, 8);
        }
    };
    // the first chunk has the row of step 0 in front
    const uint32_t front = c == 0u ? 1u : 0u;
    if (valid)
        put(lane + front, s, edge, x);
    if (front && lane == 0u) {
        const MT n1 = (MT)((uint64_t)N - 1u), v[7] = {(MT)1u, (MT)0u, n1, n1, n1, n1, n1};
        put(0u, 0u, 0u, v);
    }
    __syncthreads();
    uint8_t *dst = out + ((uint64_t)r * S + c * 64u + 1u - front) * ROW;
    const uint32_t n = (min(64u, M - c * 64u) + front) * ROW;
    const uint32_t head = (uint32_t)(-(uintptr_t)dst & 3u), words = (n - head) / 4u;
    const uint32_t tail = head + words * 4u;
    if (lane < head)
        dst[lane] = rows[lane];
    for (uint32_t i = lane; i < words; i += 64u) {
        uint32_t w;
        __builtin_memcpy(&w, rows + head + 4u * i, 4);
        ((uint32_t *)(dst + head))[i] = w;
    }
    if (tail + lane < n)
        dst[tail + lane] = rows[tail + lane];
}

// ---------------------------------------------------------------------------
// Binomial weights B(n, k; p) = C(n, k) p^k (1-p)^(n-k), the convolution
// factors of percolate/percolate.py:1067-1109, evaluated per element in FP64
// with Loader's saddle-point form (C. Loader, "Fast and Accurate Computation
// of Binomial Probabilities", 2000):
//   ln B = stirlerr(n) - stirlerr(k) - stirlerr(n-k) - bd0(k, np)
//          - bd0(n-k, nq) - ln(2 pi k (n-k) / n) / 2
// with stirlerr(m) = ln m! - ln(sqrt(2 pi m) (m/e)^m) and the deviance
// bd0(x, m) = x ln(x/m) + m - x computed without cancellation.  Only the
// window |k - np| <= 12 sigma + 48 is kept: by Bernstein's inequality each
// tail outside it holds at most exp(-72) of the mass for every sigma.  The
// window is then normalised to sum 1 as the reference normalises its array.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double stirlerr(double n)
{
    const double S0 = 1.0 / 12.0, S1 = 1.0 / 360.0, S2 = 1.0 / 1260.0,
                 S3 = 1.0 / 1680.0, S4 = 1.0 / 1188.0;
    if (n <= 15.0)
        return kStirlerr[(int)n];
    const double nn = n * n;
    return (S0 - (S1 - (S2 - (S3 - S4 / nn) / nn) / nn) / nn) / n;
}

__device__ __forceinline__ double bd0(double x, double np)
{
    if (fabs(x - np) < 0.1 * (x + np)) {
        double v = (x - np) / (x + np);
        double s = (x - np) * v;
        double ej = 2.0 * x * v;
        const double v2 = v * v;
        for (int j = 1; j < 1000; ++j) {
            ej *= v2;
            const double s1 = s + ej / (double)(2 * j + 1);
            if (s1 == s)
                return s1;
            s = s1;
        }
        return s;
    }
    return x * log(x / np) + np - x;
}

__device__ __forceinline__ double binom_pmf(double x, double n, double p)
{
    const double q = 1.0 - p;
    if (p == 0.0)
        return x == 0.0 ? 1.0 : 0.0;
    if (q == 0.0)
        return x == n ? 1.0 : 0.0;
    if (x == 0.0) {
        if (n == 0.0)
            return 1.0;
        const double lc = p < 0.1 ? -bd0(n, n * q) - n * p : n * log(q);
        return exp(lc);
    }
    if (x == n) {
        const double lc = q < 0.1 ? -bd0(n, n * p) - n * q : n * log(p);
        return exp(lc);
    }
    const double lc = stirlerr(n) - stirlerr(x) - stirlerr(n - x) -
                      bd0(x, n * p) - bd0(n - x, n * q);
    const double lf = 1.8378770664093454836 /* ln 2 pi */ + log(x) +
                      log1p(-x / n);
    return exp(lc - 0.5 * lf);
}

__global__ __launch_bounds__(256) void binom_weights_kernel(
    uint32_t n, const double *__restrict__ ps, const int64_t *__restrict__ start,
    const int64_t *__restrict__ len, int64_t kmax, double *__restrict__ w)
{
    const uint32_t pi = blockIdx.y;
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= kmax)
        return;
    double v = 0.0;
    if (k < len[pi])
        v = binom_pmf((double)(start[pi] + k), (double)n, ps[pi]);
    w[(int64_t)pi * kmax + k] = v;
}

// one block per p: divide the window by its sum
__global__ __launch_bounds__(256) void binom_normalize_kernel(
    int64_t kmax, const int64_t *__restrict__ len, double *__restrict__ w)
{
    __shared__ double part[256];
    double *row = w + (int64_t)blockIdx.x * kmax;
    const int64_t L = len[blockIdx.x];
    double acc = 0.0;
    for (int64_t k = threadIdx.x; k < L; k += 256)
        acc += row[k];
    part[threadIdx.x] = acc;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off)
            part[threadIdx.x] += part[threadIdx.x + off];
        __syncthreads();
    }
    const double total = part[0];
    if (total > 0.0)
        for (int64_t k = threadIdx.x; k < L; k += 256)
            row[k] /= total;
}

// ---------------------------------------------------------------------------
// Canonical contraction Q[p][c] = sum_k w[p][k] X[start_p + k][c] in FP64 on
// the vector ALUs: one block per p, threads stride over the window.
// ---------------------------------------------------------------------------
#define CONTRACT_MAX_COLS 32
#define PC_CONTRACT_SLICES 16

template <int C>
__global__ __launch_bounds__(256) void contract_f64_kernel(
    const double *__restrict__ x, int64_t S, int64_t x_stride,
    const int64_t *__restrict__ start, const int64_t *__restrict__ len,
    const double *__restrict__ w, int64_t kmax, double *__restrict__ out, int32_t cols)
{
    __shared__ double part[256 / 64][C];
    const uint32_t pi = blockIdx.x;
    const double *wr = w + (int64_t)pi * kmax;
    const double *xr = x + start[pi] * x_stride;
    const int64_t L = min(len[pi], S - start[pi]);   // no rows past the last
    double acc[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
        acc[c] = 0.0;
    for (int64_t k = threadIdx.x; k < L; k += 256) {
        const double wk = wr[k];
        const double *row = xr + k * x_stride;
#pragma unroll
        for (int c = 0; c < C; ++c)
            if (c < cols)
                acc[c] = fma(wk, row[c], acc[c]);
    }
    // wave reduction, then across the four waves
#pragma unroll
    for (int c = 0; c < C; ++c) {
        double v = acc[c];
        for (int off = 32; off > 0; off >>= 1)
            v += __shfl_xor(v, off, 64);
        acc[c] = v;
    }
    const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    if (lane == 0)
#pragma unroll
        for (int c = 0; c < C; ++c)
            part[wave][c] = acc[c];
    __syncthreads();
    if (threadIdx.x < (uint32_t)cols) {
        const int c = threadIdx.x;
        out[(int64_t)pi * cols + c] =
            part[0][c] + part[1][c] + part[2][c] + part[3][c];
    }
}


// ---------------------------------------------------------------------------
// Canonical contraction on the matrix cores.  One wavefront computes a tile
// of 16 p-values x 16 columns over one slice of the steps (the union of the
// 16 windows is split across blockIdx.z for parallelism); slices write
// partial sums that contract_reduce_kernel adds in a fixed order, so the
// result does not depend on scheduling.
//   FP64:   v_mfma_f64_16x16x4f64, FP64 in, FP64 accumulate.
//   FP32:   v_mfma_f32_16x16x4f32 on FP32 inputs; the FP32 accumulator is
//           added into FP64 every 8 MFMAs (bounded FP32 accumulation).
//   BF16X3: FP32 inputs split into three bf16 terms hi + mid + lo, the six
//           leading products (lo*hi, hi*lo, mid*mid, mid*hi, hi*mid,
//           hi*hi) on v_mfma_f32_16x16x32_bf16, FP32 accumulator added into
//           FP64 every 8 steps.
// Lane layout of the 16x16xK MFMAs: A row i = lane % 16 holds K/4
// consecutive k starting at (lane / 16) * K/4; B column j = lane % 16 the
// same k; register r of the output holds D[4 * (lane / 16) + r][lane % 16]
// for the FP32 accumulators and D[lane / 16 + 4 r][lane % 16] for FP64.
// ---------------------------------------------------------------------------
// Row tile of workgroup b out of T: workgroups are dealt to the 8 XCDs in
// turn, so give each XCD a contiguous run of tiles; neighbouring p-values
// read the same rows of X and then share that XCD's L2.
__device__ __forceinline__ uint32_t xcd_tile(uint32_t b, uint32_t T)
{
    const uint32_t x = b % 8u, idx = b / 8u;
    const uint32_t base = T / 8u, extra = T % 8u;
    return x * base + min(x, extra) + idx;
}

typedef double v4f64 __attribute__((ext_vector_type(4)));
typedef float v4f32 __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf16 __attribute__((ext_vector_type(8)));

#define MFMA_FLUSH 8

struct TileCtx {
    uint32_t P, C;
    int64_t x_stride, kmax;
    const int64_t *start, *len;
};

__device__ __forceinline__ int64_t tile_lo(const TileCtx &t, uint32_t p0)
{
    int64_t lo = INT64_MAX;
    for (uint32_t i = 0; i < 16 && p0 + i < t.P; ++i)
        lo = min(lo, t.start[p0 + i]);
    return lo;
}
__device__ __forceinline__ int64_t tile_hi(const TileCtx &t, uint32_t p0)
{
    int64_t hi = 0;
    for (uint32_t i = 0; i < 16 && p0 + i < t.P; ++i)
        hi = max(hi, t.start[p0 + i] + t.len[p0 + i]);
    return hi;
}

template <typename T>
__device__ __forceinline__ T load_w(const T *__restrict__ w, const TileCtx &t,
                                    uint32_t p, int64_t g)
{
    if (p >= t.P)
        return (T)0;
    const int64_t k = g - t.start[p];
    return (k >= 0 && k < t.len[p]) ? w[(int64_t)p * t.kmax + k] : (T)0;
}

template <typename T>
__device__ __forceinline__ T load_x(const T *__restrict__ x, const TileCtx &t,
                                    int64_t g, uint32_t c, int64_t S)
{
    return (c < t.C && g < S) ? x[g * t.x_stride + c] : (T)0;
}

__device__ __forceinline__ void split3(float v, __bf16 &hi, __bf16 &mid, __bf16 &lo)
{
    hi = (__bf16)v;
    const float r1 = v - (float)hi;
    mid = (__bf16)r1;
    const float r2 = r1 - (float)mid;
    lo = (__bf16)r2;
}

template <int PREC>
__global__ __launch_bounds__(64) void contract_mfma_kernel(
    const void *__restrict__ xv, int64_t S, const void *__restrict__ wv,
    TileCtx t, uint32_t slices, double *__restrict__ partial)
{
    const uint32_t lane = threadIdx.x;
    const uint32_t p0 = blockIdx.x * 16u, c0 = blockIdx.y * 16u;
    const uint32_t slice = blockIdx.z;
    const int64_t lo = tile_lo(t, p0), hi = tile_hi(t, p0);
    constexpr int64_t KSTEP = (PREC == PC_PREC_BF16X3_MFMA) ? 32 : 4;
    const int64_t steps = hi > lo ? (hi - lo + KSTEP - 1) / KSTEP : 0;
    const int64_t per = (steps + slices - 1) / slices;
    const int64_t g_begin = lo + (int64_t)slice * per * KSTEP;
    const int64_t g_end = min(hi, g_begin + per * KSTEP);
    const uint32_t i = lane % 16u, q = lane / 16u;
    const uint32_t p = p0 + i, c = c0 + i;

    double out[4] = {0.0, 0.0, 0.0, 0.0};
    if (PREC == PC_PREC_FP64_MFMA) {
        const double *w = (const double *)wv, *x = (const double *)xv;
        v4f64 acc = {0.0, 0.0, 0.0, 0.0};
        for (int64_t g = g_begin; g < g_end; g += 4) {
            const double a = load_w(w, t, p, g + q);
            const double b = load_x(x, t, g + q, c, S);
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
        }
        for (int r = 0; r < 4; ++r)
            out[r] = acc[r];
    } else if (PREC == PC_PREC_FP32_MFMA) {
        const float *w = (const float *)wv, *x = (const float *)xv;
        v4f32 acc = {0.f, 0.f, 0.f, 0.f};
        int n = 0;
        for (int64_t g = g_begin; g < g_end; g += 4) {
            const float a = load_w(w, t, p, g + q);
            const float b = load_x(x, t, g + q, c, S);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0);
            if (++n == MFMA_FLUSH) {
                for (int r = 0; r < 4; ++r)
                    out[r] += (double)acc[r];
                acc = v4f32{0.f, 0.f, 0.f, 0.f};
                n = 0;
            }
        }
        for (int r = 0; r < 4; ++r)
            out[r] += (double)acc[r];
    } else {
        const float *w = (const float *)wv, *x = (const float *)xv;
        v4f32 acc = {0.f, 0.f, 0.f, 0.f};
        int n = 0;
        for (int64_t g = g_begin; g < g_end; g += 32) {
            v8bf16 ah, am, al, bh, bm, bl;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int64_t gk = g + 8 * q + e;
                __bf16 h, m, l;
                split3(load_w(w, t, p, gk), h, m, l);
                ah[e] = h; am[e] = m; al[e] = l;
                split3(load_x(x, t, gk, c, S), h, m, l);
                bh[e] = h; bm[e] = m; bl[e] = l;
            }
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am, bm, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am, bh, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bm, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, acc, 0, 0, 0);
            if (++n == MFMA_FLUSH) {
                for (int r = 0; r < 4; ++r)
                    out[r] += (double)acc[r];
                acc = v4f32{0.f, 0.f, 0.f, 0.f};
                n = 0;
            }
        }
        for (int r = 0; r < 4; ++r)
            out[r] += (double)acc[r];
    }
    // output rows: D[4q + r][i] for the FP32-accumulating MFMAs, rows
    // interleaved as D[q + 4r][i] for v_mfma_f64_16x16x4f64
    for (int r = 0; r < 4; ++r) {
        const uint32_t row = (PREC == PC_PREC_FP64_MFMA) ? q + 4u * (uint32_t)r
                                                         : 4u * q + (uint32_t)r;
        const uint32_t pr = p0 + row, cc = c0 + i;
        if (pr < t.P && cc < t.C)
            partial[((int64_t)slice * t.P + pr) * t.C + cc] = out[r];
    }
}

// Wide contraction on the FP64 matrix cores, for many columns (the per-run
// canonical statistics of a whole chunk of runs at once): a GEMM of the
// banded weights with X.  Workgroup of 4 wavefronts on a tile of 64 p x TC
// columns; wave w takes the p rows 16w..16w+15 and all TC columns, TC / 16
// v_mfma_f64_16x16x4f64 accumulators sharing the weight operand.  The steps
// of the union of the tile's 64 windows advance 16 at a time: the 16 x TC
// block of X is staged through LDS (double-buffered, one barrier per block),
// each lane's 4 weights are consecutive steps, and a wave leaves out the
// blocks that none of its 16 windows meets.  Partial sums of K-slices
// (blockIdx.y) go to `dst` + slice * P * C and contract_reduce_kernel adds
// them in order.
//
// Blocks lie on multiples of 16 steps and every tile goes round its own
// blocks from the one that is 0 modulo their number, so that tiles of
// neighbouring p, which share most of their steps, read the same rows of X
// at about the same time; tiles are dealt XCD-contiguous in column-major
// order, so they also share an L2.  1000 p, windows of 2260 steps, 21504
// columns: 1.94 ms, against 2.46 with every tile starting at its own window
// (the X rows then came from beyond the L2, 4.7 TB/s of them) and 65 vector
// instructions a block of 16 MFMAs instead of 12; the MFMAs alone take 1.55.
// 128 p a tile took 1.97 ms, 128 columns 1.91, both 2.08.
// Where the p are few and far apart, every block lies outside some row's
// window, and the weights put in place one by one in each of them held up the
// MFMAs: 16 p in 0.1, n = 32512, 64 columns 33.4 us, now (only in the blocks
// where a lane's four are cut, 9 % of them, and by two rotations) 26.8; with
// n = 130560 87 and 65.
#define WIDE_TILE 64
#define WIDE_KSTEP 16

typedef double v2d8 __attribute__((ext_vector_type(2), aligned(8)));

// The caller has at least TC columns.
template <int TC>
__global__ __launch_bounds__(256) void contract_wide_f64_kernel(
    const double *__restrict__ x, int64_t S, const double *__restrict__ w,
    TileCtx t, uint32_t tiles_p, uint32_t slices, double *__restrict__ dst)
{
    constexpr int KS = WIDE_KSTEP, STRIDE = TC + 4, NJ = TC / 16, E = TC / 16;
    __shared__ double xs[2][KS * STRIDE];
    __shared__ int32_t range[2][4];
    const uint32_t tile = xcd_tile(blockIdx.x, gridDim.x);
    const uint32_t p0 = (tile % tiles_p) * WIDE_TILE;
    // the last tile ends at the last column and shares some with the one before
    const uint32_t c0 = min((tile / tiles_p) * TC, t.C - TC);
    const uint32_t slice = blockIdx.y;
    const uint32_t tid = threadIdx.x, wave = uniform(tid / 64u), lane = tid % 64u;
    const uint32_t i = lane % 16u, q = lane / 16u;

    // the lane's row of weights; the steps of an X that fits memory fit 31
    // bits
    const uint32_t p = p0 + wave * 16u + i;
    const bool prow = p < t.P;
    const int32_t wstart = prow ? (int32_t)t.start[p] : 0, wlen = prow ? (int32_t)t.len[p] : 0;
    const double *wrow = w + (int64_t)(prow ? p : 0) * t.kmax;
    // four weights are read at a time, those of a shorter window apart
    const int32_t wlast = max(wlen - 4, 0);
    const double *wfour = wlen < 4 ? x : wrow;
    const bool any_short = ballot(wlen > 0 && wlen < 4) != 0u;
    // union and intersection of the wave's windows
    int32_t any_lo = wlen > 0 ? wstart : INT32_MAX, any_hi = wlen > 0 ? wstart + wlen : 0;
    int32_t all_lo = wstart, all_hi = wstart + wlen;
    for (int off = 8; off > 0; off >>= 1) {
        any_lo = min(any_lo, __shfl_xor(any_lo, off, 64));
        any_hi = max(any_hi, __shfl_xor(any_hi, off, 64));
        all_lo = max(all_lo, __shfl_xor(all_lo, off, 64));
        all_hi = min(all_hi, __shfl_xor(all_hi, off, 64));
    }
    any_lo = (int32_t)uniform((uint32_t)any_lo);
    any_hi = (int32_t)uniform((uint32_t)any_hi);
    all_lo = (int32_t)uniform((uint32_t)all_lo);
    all_hi = (int32_t)uniform((uint32_t)all_hi);
    if (lane == 0) {
        range[0][wave] = any_lo;
        range[1][wave] = any_hi;
    }
    __syncthreads();
    int32_t lo = INT32_MAX, hi = 0;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        lo = min(lo, range[0][v]);
        hi = max(hi, range[1][v]);
    }
    lo = (int32_t)uniform((uint32_t)lo);
    hi = (int32_t)uniform((uint32_t)min((int64_t)hi, S));
    // the slice's blocks [first, first + count)
    int32_t first = 0, count = 0;
    if (lo < hi) {
        const int32_t b0 = lo / KS, all = (hi + KS - 1) / KS - b0;
        const int32_t per = (all + (int32_t)slices - 1) / (int32_t)slices;
        first = b0 + (int32_t)slice * per;
        count = max(min(b0 + all, first + per) - first, 0);
    }

    v4f64 acc[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
        acc[j] = v4f64{0.0, 0.0, 0.0, 0.0};

    // X loader: thread tid reads row tid / 16 of the block, columns
    // tid % 16 + 16 e.  Loads are issued whether needed or not, from clamped
    // places, so that no wait stands between them and the step they overlap.
    const uint32_t lr = tid / 16u, lc = tid % 16u;
    const double *xlane = x + (int64_t)lr * t.x_stride + (c0 + lc);
    const double *xlast = x + (S - 1) * t.x_stride + (c0 + lc);
    auto load_b = [&](int32_t blk, double *b) {
        const double *row = xlane + (int64_t)(blk * KS) * t.x_stride;
        if (blk * KS + KS > (int32_t)S)
            row = row < xlast ? row : xlast;
#pragma unroll
        for (int e = 0; e < E; ++e)
            b[e] = row[16 * e];
    };
    // into LDS, rows outside the tile's steps as 0
    auto store_b = [&](int32_t blk, int buf, double *b) {
        if (blk * KS < lo || blk * KS + KS > hi) {
            const int32_t row = blk * KS + (int32_t)lr;
            const bool ok = row >= lo && row < hi;
#pragma unroll
            for (int e = 0; e < E; ++e)
                b[e] = ok ? b[e] : 0.0;
        }
#pragma unroll
        for (int e = 0; e < E; ++e)
            xs[buf][lr * STRIDE + lc + 16 * e] = b[e];
    };
    // four weights of consecutive steps a lane, from the nearest four of its
    // window; step() puts them in place where a window starts or ends
    auto load_a = [&](int32_t blk, v2d8 *a) {
        const int32_t k = blk * KS + 4 * (int32_t)q - wstart;
        const double *at = wfour + min(max(k, 0), wlast);
        a[0] = *(const v2d8 *)at;
        a[1] = *(const v2d8 *)(at + 2);
    };
    // columns of a tile: lane i of accumulator j holds 32 (j / 2) + 2 i + j % 2
    auto step = [&](int32_t blk, int32_t nxt, int buf, const v2d8 *a, v2d8 *an, bool more) {
        double b[E];
        load_b(nxt, b);
        load_a(nxt, an);
        const double *xb = xs[buf] + 4u * q * STRIDE + 2u * i;
        if (blk * KS < any_hi && (blk + 1) * KS > any_lo) {
            double av[4] = {a[0][0], a[0][1], a[1][0], a[1][1]};
            if (blk * KS < all_lo || blk * KS + KS > all_hi) {
                const int32_t k = blk * KS + 4 * (int32_t)q - wstart;
                const bool whole = k >= 0 && k + 4 <= wlen;
                if (ballot(!whole && k > -4 && k < wlen)) {
                    // some lane's four steps are partly in its window: the
                    // weight of step e is at e + d, or (short) read by itself
                    const int32_t d = k - min(max(k, 0), wlast);
                    const double v[4] = {av[0], av[1], av[2], av[3]};
                    double by1[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        by1[e] = d & 1 ? v[(e + 1) & 3] : v[e];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const bool in = (uint32_t)(k + e) < (uint32_t)wlen;
                        av[e] = d & 2 ? by1[(e + 2) & 3] : by1[e];
                        av[e] = in ? av[e] : 0.0;
                        if (any_short && in)
                            av[e] = wrow[k + e];
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        av[e] = whole ? av[e] : 0.0;
                }
            }
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
#pragma unroll
                for (int j = 0; j < NJ; ++j)
                    acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                        av[kk], xb[kk * STRIDE + 32 * (j / 2) + (j & 1)], acc[j], 0, 0, 0);
        }
        if (more)
            store_b(nxt, buf ^ 1, b);
        __syncthreads();
    };
    if (count > 0) {
        int32_t at = (count - first % count) % count;
        auto advance = [&]() {
            const int32_t blk = first + at;
            at = at + 1 == count ? 0 : at + 1;
            return blk;
        };
        v2d8 a0[2], a1[2];
        double b[E];
        int32_t cur = advance();
        load_b(cur, b);
        load_a(cur, a0);
        store_b(cur, 0, b);
        __syncthreads();
        int32_t n = 0;
        for (; n + 2 <= count; n += 2) {
            const int32_t nxt = advance();
            step(cur, nxt, 0, a0, a1, true);
            cur = advance();
            step(nxt, cur, 1, a1, a0, true);
        }
        if (n < count)
            step(cur, cur, 0, a0, a1, false);
    }
    // register r of accumulator j holds D[q + 4r][i] of column block j
    double *out = dst + (int64_t)slice * t.P * t.C;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t row = p0 + wave * 16u + q + 4u * (uint32_t)r;
            const uint32_t c = c0 + 32u * (uint32_t)(j / 2) + 2u * i + (uint32_t)(j & 1);
            if (row < t.P)
                out[(int64_t)row * t.C + c] = acc[j][r];
        }
}

__global__ __launch_bounds__(256) void contract_reduce_kernel(
    const double *__restrict__ partial, uint32_t slices, int64_t n,
    double *__restrict__ out)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n)
        return;
    double acc = 0.0;
    for (uint32_t s = 0; s < slices; ++s)
        acc += partial[(int64_t)s * n + i];
    out[i] = acc;
}

__global__ __launch_bounds__(256) void f64_to_f32_kernel(
    const double *__restrict__ in, int64_t n, float *__restrict__ out)
{
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * 256)
        out[i] = (float)in[i];
}

// ---------------------------------------------------------------------------
// Canonical averages with the binomial weights generated inside the
// contraction (no weight matrix in HBM):
//   out[p][c] = sum_k B(n, k; p) X[k][c] / sum_k B(n, k; p)
// over the window of p.  The normaliser is the contraction of a virtual
// all-ones column C, so it goes through the same arithmetic as the columns.
//
// Tiles: one wavefront = 16 p-values x 16 columns (column C is the ones
// column) over one of `slices` pieces of the union of the 16 windows.  The
// four lane groups q = lane / 16 each walk a contiguous quarter of the piece,
// one k per MFMA k-position, so every lane's weights form a sequence of
// consecutive k: one direct evaluation (Loader's form, binom_pmf) where the
// sequence enters the window, then the exact ratio
//   B(n, k; p) / B(n, k - 1; p) = (n - k + 1) / k * p / (1 - p),
// with a fresh direct evaluation every FUSED_REANCHOR steps, so the
// relative error stays below about 1e-13.  The MFMA's k positions only have
// to agree between the A (weights) and B (columns) operands, which they do
// because lane (i, q) supplies both for the same k.
//
// SPLIT_BF16 (Ozaki-style exact split): per window of 64 k (16 consecutive
// k in each lane group), a weight is scaled by 2^(32 - E), E per row
// (max w < 2^E over the row's 64 weights of the window), and a column value
// by 2^(32 - F), F per column (max |x| < 2^F), rounded to 32-bit integers and
// cut into four bytes, most significant first.  Bytes are exact in bf16 and
// their products (< 2^16) exact in FP32; the 13 byte-pair products with
// s + t <= 4 run on v_mfma_f32_16x16x32_bf16, one FP32 accumulator per level
// s + t.  Within a window each level sums at most 4 x 64 products of at most
// 255 x 255, below 2^24, so the FP32 sums are exact integers; they are added
// into FP64 scaled by 2^(E + F - 16 - 8 (s + t)).  Scales per window keep
// the far tails of the weights (and small column values) at full relative
// precision; the dropped levels and the rounding of the 32-bit integers
// leave a relative error near 1e-10 for non-negative columns.
// ---------------------------------------------------------------------------
// Bound by issue: a step is an FP64 MFMA of 64 cycles and, where no row's
// window starts or ends, about seven vector instructions beside it (two
// products, the ratio's broadcast, the load).  L = 1024, 4096 p in [0.3,
// 0.7], 14 columns: 100 us, 127 with lane shuffles and window tests in every
// step; the MFMAs alone take 35.
#define FUSED_REANCHOR 1024
#define FUSED_F64_UNROLL 8

struct FusedCtx {
    const double *x;
    int64_t x_stride;
    const double *ps;
    const int64_t *start, *len;
    uint32_t n, P, C;
};

// Direct evaluations in the walks are rare (one per lane and range, and one
// per FUSED_REANCHOR steps): kept out of line so the contraction loops keep
// their registers (112 instead of 160 VGPRs, 4 waves per SIMD).
__device__ __attribute__((noinline)) double binom_pmf_outline(double x, double n,
                                                               double p)
{
    return binom_pmf(x, n, p);
}

// Per-lane walk over consecutive k of one row's weights.
struct BinomWalk {
    double n, p, pq, w, anchor;
    int64_t ka, kend; // in-window k of this lane's range: [ka, kend)
};

__device__ __forceinline__ void walk_init(BinomWalk &b, const FusedCtx &f,
                                          uint32_t row, int64_t k0, int64_t k1)
{
    b.n = (double)f.n;
    b.p = 0.5;
    int64_t st = 0, ln = 0;
    if (row < f.P) {
        b.p = f.ps[row];
        st = f.start[row];
        ln = f.len[row];
        // the degenerate distributions hold all their mass at one k
        if (b.p <= 0.0) {
            st = 0;
            ln = 1;
        } else if (b.p >= 1.0) {
            st = (int64_t)f.n;
            ln = 1;
        }
    }
    // (all mass at k = n when p is 1: no recursion)
    b.pq = b.p >= 1.0 ? 0.0 : b.p / (1.0 - b.p);
    b.ka = max(k0, st);
    b.kend = min(k1, st + ln);
    b.anchor = b.ka < b.kend ? binom_pmf_outline((double)b.ka, b.n, b.p) : 0.0;
    b.w = 0.0;
}

// Weight at k (k advances by one per call) from the weight at k - 1 and
// ratio = (n - k + 1) / k; `fresh` replaces the ratio step by a direct
// evaluation (a uniform branch every FUSED_REANCHOR steps).
__device__ __forceinline__ double walk_step(BinomWalk &b, int64_t k, bool fresh,
                                            double ratio)
{
    double v;
    if (fresh && k > b.ka && k < b.kend)
        v = binom_pmf_outline((double)k, b.n, b.p);
    else
        v = b.w * ratio * b.pq;
    v = (k == b.ka) ? b.anchor : v;
    b.w = v;
    return (k >= b.ka && k < b.kend) ? v : 0.0;
}

__device__ __forceinline__ double fused_x(const FusedCtx &f, int64_t k, uint32_t c)
{
    if (c < f.C)
        return f.x[k * f.x_stride + c];
    return c == f.C ? 1.0 : 0.0;
}

// K-range of this wave: the union of the tile's windows, cut into `slices`
// pieces of a multiple of `quant` steps; returns false if the piece is empty.
__device__ __forceinline__ bool fused_range(const FusedCtx &f, uint32_t p0,
                                            uint32_t slices, uint32_t slice,
                                            int64_t quant, int64_t &g_begin,
                                            int64_t &g_end, int64_t &per)
{
    // a lane per row, then the extremes over the rows of 16 lanes (all alike)
    int64_t lo = INT64_MAX, hi = 0;
    const uint32_t row = p0 + threadIdx.x % 16u;
    if (row < f.P) {
        const double p = f.ps[row];
        int64_t st = f.start[row], ln = f.len[row];
        if (p <= 0.0) {
            st = 0;
            ln = 1;
        } else if (p >= 1.0) {
            st = (int64_t)f.n;
            ln = 1;
        }
        lo = st;
        hi = st + ln;
    }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) {
        lo = min(lo, (int64_t)__shfl_xor((long long)lo, off, 64));
        hi = max(hi, (int64_t)__shfl_xor((long long)hi, off, 64));
    }
    lo = (int64_t)read_lane((uint64_t)lo, 0u);
    hi = (int64_t)read_lane((uint64_t)hi, 0u);
    if (hi <= lo)
        return false;
    per = (hi - lo + slices - 1) / slices;
    per = (per + quant - 1) / quant * quant;
    g_begin = lo + (int64_t)slice * per;
    g_end = min(hi, g_begin + per);
    return g_begin < g_end;
}

static __device__ const double kOnes = 1.0;

// Lanes FIRST .. FIRST + 7 of every row of 16 lanes, each to its whole row.
template <int LANE>
__device__ __forceinline__ double row_lane(double v)
{
    const uint64_t w = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)w, 0x150 + LANE, 0xf, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(w >> 32), 0x150 + LANE, 0xf, 0xf, false);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
template <int FIRST>
__device__ __forceinline__ void row_lanes(double v, double (&out)[FUSED_F64_UNROLL])
{
    static_assert(FUSED_F64_UNROLL == 8, "eight lanes");
    out[0] = row_lane<FIRST>(v);
    out[1] = row_lane<FIRST + 1>(v);
    out[2] = row_lane<FIRST + 2>(v);
    out[3] = row_lane<FIRST + 3>(v);
    out[4] = row_lane<FIRST + 4>(v);
    out[5] = row_lane<FIRST + 5>(v);
    out[6] = row_lane<FIRST + 6>(v);
    out[7] = row_lane<FIRST + 7>(v);
}

__global__ __launch_bounds__(64, 3) void canonical_fused_f64_kernel(
    FusedCtx f, uint32_t slices, double *__restrict__ partial)
{
    const uint32_t lane = threadIdx.x, i = lane % 16u, q = lane / 16u;
    const uint32_t p0 = xcd_tile(blockIdx.x, gridDim.x) * 16u;
    const uint32_t c0 = blockIdx.y * 16u, slice = blockIdx.z;
    const uint32_t C1 = f.C + 1u, c = c0 + i;
    int64_t g_begin = 0, g_end = 0, per = 0;
    v4f64 acc0 = {0.0, 0.0, 0.0, 0.0}, acc1 = {0.0, 0.0, 0.0, 0.0};
    if (fused_range(f, p0, slices, slice, 4 * FUSED_F64_UNROLL, g_begin, g_end, per)) {
        const int64_t Lq = per / 4;
        const int64_t kq0 = g_begin + (int64_t)q * Lq;
        const int64_t kq1 = min(kq0 + Lq, g_end);
        BinomWalk b;
        walk_init(b, f, p0 + i, kq0, kq1);
        // the ratio (n - k + 1) / k depends on k only, shared by the 16 rows
        // of a lane group: each lane divides once per 16 steps, for step
        // j0 + lane % 16 of group lane / 16, and a step takes it from the
        // lane of its row with a DPP broadcast
        double rr = 0.0;
        // Columns one chunk ahead: column C reads a 1 over and over, lanes past
        // it column 0 (their outputs are not kept); steps past the lane's
        // range count as 0.
        const double *xc = c == f.C ? &kOnes : f.x + (c < f.C ? c : 0u);
        const int64_t stride = c == f.C ? 0 : f.x_stride;
        const int64_t kl = max(kq1 - 1, (int64_t)0);
        // the row's window within the lane's range, as steps of the walk
        const int ja = (int)min(b.ka - kq0, (int64_t)1 << 30);
        const int je = (int)min(max(b.kend - kq0, (int64_t)0), (int64_t)1 << 30);
        // A chunk before this step ends no window: the one that does, at its
        // last step too, has to clear the weight.  (Where the lane's range
        // ends as well, or first, the steps after it count as 0 anyway.)
        const int jw = b.kend == kq1 ? je + 1 : je;
        double xn[FUSED_F64_UNROLL];
        // FULL: the next chunk lies in every lane's range.  (Both forms of
        // loads in one loop would be branches, whose loads are waited for
        // where the branches meet.)
        auto chunk = [&](int64_t j0, auto full) __attribute__((always_inline)) {
            constexpr bool FULL = decltype(full)::value;
            double a[FUSED_F64_UNROLL], x[FUSED_F64_UNROLL];
            const int64_t k0 = kq0 + j0, k1 = k0 + FUSED_F64_UNROLL;
            const double *next = xc + k1 * stride;
#pragma unroll
            for (int u = 0; u < FUSED_F64_UNROLL; ++u) {
                x[u] = xn[u];
                if (!FULL) {
                    x[u] = k0 + u < kq1 ? x[u] : 0.0;
                    next = xc + min(k1 + u, kl) * stride;
                }
                xn[u] = *next;
                if (FULL)
                    next += stride;
            }
            if ((j0 & 15) == 0) {
                const int64_t kr = g_begin + (int64_t)(lane / 16u) * Lq + j0 + (lane % 16u);
                rr = kr ? (b.n - (double)kr + 1.0) / (double)kr : 0.0;
            }
            double ratio[FUSED_F64_UNROLL];
            if (j0 & 8)
                row_lanes<8>(rr, ratio);
            else
                row_lanes<0>(rr, ratio);
            const bool fresh = j0 > 0 && j0 % FUSED_REANCHOR == 0;
            // where no row's window starts or ends in the chunk, a step is the
            // two products alone: rows before their window, past it, or past P
            // hold weight 0 (past a window that their range of steps cuts
            // short, they meet columns of 0)
            const int j = (int)j0;
            double direct = 0.0;
            const bool anew = fresh && j > ja && j < je;
            if (anew)
                direct = binom_pmf_outline((double)k0, b.n, b.p);
            const double w0 = b.w * ratio[0] * b.pq;
            b.w = anew ? direct : w0;
            const bool before = j + FUSED_F64_UNROLL <= ja;
            if (ballot(before || j >= je || (j > ja && j + FUSED_F64_UNROLL < jw)) == ~0ull) {
                a[0] = b.w;
#pragma unroll
                for (int u = 1; u < FUSED_F64_UNROLL; ++u)
                    a[u] = b.w = b.w * ratio[u] * b.pq;
            } else {
#pragma unroll
                for (int u = 0; u < FUSED_F64_UNROLL; ++u) {
                    if (u)
                        b.w = b.w * ratio[u] * b.pq;
                    b.w = j + u == ja ? b.anchor : b.w;
                    a[u] = j + u >= ja && j + u < je ? b.w : 0.0;
                }
                if (before || j + FUSED_F64_UNROLL >= je)
                    b.w = 0.0;
            }
#pragma unroll
            for (int u = 0; u < FUSED_F64_UNROLL; u += 2) {
                acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u], x[u], acc0, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u + 1], x[u + 1], acc1, 0, 0, 0);
            }
        };
#pragma unroll
        for (int u = 0; u < FUSED_F64_UNROLL; ++u)
            xn[u] = xc[min(kq0 + u, kl) * stride];
        // the last lane group has the shortest range
        const int64_t jf = min(Lq, g_end - g_begin - 3 * Lq) - 2 * FUSED_F64_UNROLL;
        int64_t j0 = 0;
        for (; j0 <= jf; j0 += FUSED_F64_UNROLL)
            chunk(j0, std::true_type());
        for (; j0 < Lq; j0 += FUSED_F64_UNROLL)
            chunk(j0, std::false_type());
    }
    // v_mfma_f64_16x16x4f64: register r holds D[q + 4r][i]
    for (int r = 0; r < 4; ++r) {
        const uint32_t row = p0 + q + 4u * (uint32_t)r;
        if (row < f.P && c < C1)
            partial[((int64_t)slice * f.P + row) * C1 + c] = acc0[r] + acc1[r];
    }
}

// |v| 2^e rounded to a 32-bit integer (e makes |v| 2^e < 2^32)
__device__ __forceinline__ uint32_t split_u32(double v, int e)
{
    return (uint32_t)fmin(ldexp(fabs(v), e) + 0.5, 4294967295.0);
}

// byte `s` (0 = most significant) of u as a bf16, negated when neg
__device__ __forceinline__ __bf16 byte_bf16(uint32_t u, int s, bool neg)
{
    const float v = (float)((u >> (24 - 8 * s)) & 255u);
    return (__bf16)(neg ? -v : v);
}

__global__ __launch_bounds__(64) void canonical_fused_split_kernel(
    FusedCtx f, uint32_t slices, double *__restrict__ partial)
{
    const uint32_t lane = threadIdx.x, i = lane % 16u, q = lane / 16u;
    const uint32_t p0 = xcd_tile(blockIdx.x, gridDim.x) * 16u;
    const uint32_t c0 = blockIdx.y * 16u, slice = blockIdx.z;
    const uint32_t C1 = f.C + 1u, c = c0 + i;
    int64_t g_begin = 0, g_end = 0, per = 0;
    double out[4] = {0.0, 0.0, 0.0, 0.0};
    if (fused_range(f, p0, slices, slice, 64, g_begin, g_end, per)) {
        const int64_t Lq = per / 4;
        const int64_t kq0 = g_begin + (int64_t)q * Lq;
        const int64_t kq1 = min(kq0 + Lq, g_end);
        BinomWalk b;
        walk_init(b, f, p0 + i, kq0, kq1);
        for (int64_t j0 = 0; j0 < Lq; j0 += 16) {
            double x[16], w[16];
            double m = 0.0;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int64_t k = kq0 + j0 + e;
                x[e] = k < kq1 ? fused_x(f, k, c) : 0.0;
                m = fmax(m, fabs(x[e]));
            }
            const bool fresh = j0 > 0 && j0 % FUSED_REANCHOR == 0;
            // one division per lane per window: the ratio (n - k + 1) / k
            // for step j0 + lane % 16 of group lane / 16, read back by the
            // 16 rows of each group with a lane shuffle
            const int64_t kr = g_begin + (int64_t)(lane / 16u) * Lq + j0 + (lane % 16u);
            const double rr = (b.n - (double)kr + 1.0) / (double)kr;
            double wm = 0.0;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const double ratio = __shfl(rr, (int)(q * 16u) + e, 64);
                w[e] = walk_step(b, kq0 + j0 + e, fresh && e == 0, ratio);
                wm = fmax(wm, w[e]);
            }
            // scales of column i and row i over the window: lanes i, i+16,
            // i+32, i+48 hold its four runs of 16 k
            m = fmax(m, __shfl_xor(m, 16, 64));
            m = fmax(m, __shfl_xor(m, 32, 64));
            wm = fmax(wm, __shfl_xor(wm, 16, 64));
            wm = fmax(wm, __shfl_xor(wm, 32, 64));
            const int F = m > 0.0 ? ilogb(m) + 1 : 0;
            const int Ew = wm > 0.0 ? ilogb(wm) + 1 : 0;
            // output register r holds row 4q + r: its scale from lane 4q + r
            int Er[4];
#pragma unroll
            for (int r = 0; r < 4; ++r)
                Er[r] = __shfl(Ew, (int)(4u * q) + r, 64);
            v4f32 acc[5];
#pragma unroll
            for (int l = 0; l < 5; ++l)
                acc[l] = v4f32{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                v8bf16 A[4], B[4];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const uint32_t uw = split_u32(w[8 * h + e], 32 - Ew);
                    const uint32_t ux = split_u32(x[8 * h + e], 32 - F);
                    const bool neg = x[8 * h + e] < 0.0;
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        A[s][e] = byte_bf16(uw, s, false);
                        B[s][e] = byte_bf16(ux, s, neg);
                    }
                }
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        if (s + t <= 4)
                            acc[s + t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                A[s], B[t], acc[s + t], 0, 0, 0);
            }
#pragma unroll
            for (int l = 0; l < 5; ++l)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    out[r] += ldexp((double)acc[l][r], Er[r] + F - 16 - 8 * l);
        }
    }
    // FP32-accumulating MFMA: register r holds D[4q + r][i]
    for (int r = 0; r < 4; ++r) {
        const uint32_t row = p0 + 4u * q + (uint32_t)r;
        if (row < f.P && c < C1)
            partial[((int64_t)slice * f.P + row) * C1 + c] = out[r];
    }
}

// out[p][c] = sum over slices of partial[.][p][c] / the same sum of the
// ones column, in a fixed order
__global__ __launch_bounds__(256) void fused_reduce_kernel(
    const double *__restrict__ partial, uint32_t slices, uint32_t P, uint32_t C,
    double *__restrict__ out)
{
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (int64_t)P * C)
        return;
    const int64_t p = idx / C, c = idx % C;
    const uint32_t C1 = C + 1u;
    double num = 0.0, den = 0.0;
    const double *row = partial + p * C1;
    const int64_t step = (int64_t)P * C1;
    uint32_t s = 0;
    for (; s + 8u <= slices; s += 8u) {
        // eight slices' loads in flight, added in order
        double v[8], w[8];
#pragma unroll
        for (uint32_t u = 0; u < 8u; ++u) {
            v[u] = row[(s + u) * step + c];
            w[u] = row[(s + u) * step + C];
        }
#pragma unroll
        for (uint32_t u = 0; u < 8u; ++u) {
            num += v[u];
            den += w[u];
        }
    }
    for (; s < slices; ++s) {
        num += row[s * step + c];
        den += row[s * step + C];
    }
    out[idx] = num / den;
}


// ---------------------------------------------------------------------------
// Per-run observables as FP64 columns over a window of steps, the input of
// the per-run canonical statistics (percolate/hpc.py:496-512):
// out[(s - g_lo) * (R * C) + r * C + c] for steps s in [g_lo, g_lo + g_len),
// columns [has_spanning_cluster if spanning,] max_cluster_size,
// moments[0..4] (moments as their uint64 values, like the reference's
// structured array).
// ---------------------------------------------------------------------------
// 3072 runs of L = 128 over 5600 steps, 0.96 GB of columns: 0.30 ms with four
// runs a workgroup (two 0.45, eight 0.38), 0.37 with a record at a time and one
// row a store; a copy writes that much in 0.2.
#define WT_RUNS 4u

template <typename RecT, bool WIDE>
__global__ __launch_bounds__(64) void window_traces_kernel(
    uint32_t N, uint32_t M, uint32_t R, const RecT *__restrict__ records,
    int64_t rec_stride, const uint32_t *__restrict__ span_step,
    const uint64_t *__restrict__ chunk_state, int64_t g_lo, int64_t g_len,
    int spanning, double *__restrict__ out)
{
    // Block (chunk of 64 steps, group of WT_RUNS runs): lane = step while
    // the observables are computed, then the tile goes out row by row, the
    // group's WT_RUNS * cols values of a step contiguous in the output (one
    // coalesced store per step instead of 64 scattered ones per run)
    using MT = typename Wide<WIDE>::T;
    __shared__ double tile[64][WT_RUNS * 7];
    const uint32_t lane = threadIdx.x;
    const uint32_t r0 = blockIdx.y * WT_RUNS;
    const uint32_t nr = min((uint32_t)WT_RUNS, R - r0);
    const uint32_t C = (M + 63u) / 64u;
    // chunk index of this block within the steps 1..M (state after c*64)
    const int64_t first_chunk = g_lo > 0 ? (g_lo - 1) / 64 : 0;
    const int64_t c = first_chunk + blockIdx.x;
    const int cols = spanning ? 7 : 6;
    const int64_t width = (int64_t)R * cols;
    if (c >= (int64_t)C) {
        // steps past M cannot exist; only step 0 needs the no-edge case
        return;
    }
    const int64_t q = c * 64 + lane; // record index, step q + 1
    const bool valid = q < (int64_t)M;
    // every run's record before the first is used (past the end the last's)
    RecT recs[WT_RUNS];
#pragma unroll
    for (uint32_t j = 0; j < WT_RUNS; ++j)
        recs[j] = records[(int64_t)min(r0 + j, R - 1u) * rec_stride + min(q, (int64_t)M - 1)];
#pragma unroll
    for (uint32_t j = 0; j < WT_RUNS; ++j) {
        if (j >= nr)
            break;
        const uint32_t r = r0 + j;
        const RunState<WIDE> st0 = load_state<WIDE>(
            chunk_state + ((size_t)r * C + (size_t)c) * PC_STATE_WORDS);
        const RecT rec = valid ? recs[j] : (RecT)0;
        const RunState<WIDE> st = advance<WIDE>(st0, Deltas<WIDE>(rec));
        MT x[7];
        observables<WIDE>(st, N, (uint64_t)(q + 1) >= span_step[r], x);
        double *row = tile[lane] + j * cols;
        int k = 0;
        if (spanning)
            row[k++] = (double)(uint32_t)x[1];
        // the largest cluster, the clusters and the sites beside it: 32 bits
        row[k++] = (double)(uint32_t)x[0];
        row[k++] = (double)(uint32_t)x[2];
        row[k++] = (double)(uint32_t)x[3];
        for (int m = 2; m < 5; ++m)
            row[k++] = (double)(uint64_t)x[2 + m];
    }
    __syncthreads();
    // as many rows at a time as the lanes hold
    const uint32_t n = nr * (uint32_t)cols, rows = 64u / n;
    const uint32_t first_row = lane / n, col = lane % n;
    if (first_row < rows)
        for (uint32_t i = first_row; i < 64u; i += rows) {
            const int64_t step = c * 64 + i + 1;
            if (step <= (int64_t)M && step >= g_lo && step < g_lo + g_len)
                out[(step - g_lo) * width + (int64_t)r0 * cols + col] = tile[i][col];
        }
    if (c == first_chunk && g_lo == 0 && lane < nr) {
        // step 0: max 1, no spanning, moments N - 1
        double *row = out + (int64_t)(r0 + lane) * cols;
        int k = 0;
        if (spanning)
            row[k++] = 0.0;
        row[k++] = 1.0;
        for (int m = 0; m < 5; ++m)
            row[k++] = (double)((uint64_t)N - 1u);
    }
}

// Mean and sum of squared deviations over runs of q[p][r * cols + c]
// (two passes, fixed order): the (n, mean, M2) of percolate/hpc.py:561-702.
// One workgroup per p reads that p's contiguous row of R * cols values:
// thread t takes runs t, t + 256, ... (cols consecutive values each), and
// the 256 partial sums of a column meet in a fixed LDS tree, so the result
// does not depend on scheduling.
#define RUN_MOMENTS_COLS 8

__device__ __forceinline__ double block_sum_256(double v, double *red)
{
    // fixed-order tree: wave-local butterfly, then the 4 wave totals in order
    for (int off = 32; off > 0; off >>= 1)
        v += __shfl_xor(v, off, 64);
    const uint32_t wave = threadIdx.x / 64;
    __syncthreads();
    if (threadIdx.x % 64 == 0)
        red[wave] = v;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}

__global__ __launch_bounds__(256) void run_moments_kernel(
    const double *__restrict__ q, uint32_t P, uint32_t R, uint32_t cols,
    double *__restrict__ mean, double *__restrict__ m2)
{
    __shared__ double red[4];
    const uint32_t p = blockIdx.x;
    const double *row = q + (uint64_t)p * R * cols;
    double s[RUN_MOMENTS_COLS];
#pragma unroll
    for (int c = 0; c < RUN_MOMENTS_COLS; ++c)
        s[c] = 0.0;
    for (uint32_t r = threadIdx.x; r < R; r += 256) {
#pragma unroll
        for (int c = 0; c < RUN_MOMENTS_COLS; ++c)
            if (c < (int)cols)
                s[c] += row[(uint64_t)r * cols + c];
    }
    double mu[RUN_MOMENTS_COLS];
#pragma unroll
    for (int c = 0; c < RUN_MOMENTS_COLS; ++c)
        mu[c] = c < (int)cols ? block_sum_256(s[c], red) / (double)R : 0.0;
#pragma unroll
    for (int c = 0; c < RUN_MOMENTS_COLS; ++c)
        s[c] = 0.0;
    for (uint32_t r = threadIdx.x; r < R; r += 256) {
#pragma unroll
        for (int c = 0; c < RUN_MOMENTS_COLS; ++c)
            if (c < (int)cols) {
                const double d = row[(uint64_t)r * cols + c] - mu[c];
                s[c] = fma(d, d, s[c]);
            }
    }
#pragma unroll
    for (int c = 0; c < RUN_MOMENTS_COLS; ++c) {
        if (c < (int)cols) {
            const double d2 = block_sum_256(s[c], red);
            if (threadIdx.x == 0) {
                mean[(uint64_t)p * cols + c] = mu[c];
                m2[(uint64_t)p * cols + c] = d2;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Microcanonical mean and sample standard deviation from the exact sums:
// mean = S1 / R, std = sqrt((R S2 - S1^2) / (R (R - 1))), with the numerator
// formed exactly in 256-bit integers before the single rounding to FP64.
// ---------------------------------------------------------------------------
struct u256 {
    uint64_t w[4];
};

__device__ __forceinline__ u256 mul_u192_u64(const uint64_t a[3], uint64_t b)
{
    u256 r;
    u128 carry = 0;
    for (int i = 0; i < 3; ++i) {
        const u128 t = (u128)a[i] * b + carry;
        r.w[i] = (uint64_t)t;
        carry = t >> 64;
    }
    r.w[3] = (uint64_t)carry;
    return r;
}

__device__ __forceinline__ u256 square_u128(uint64_t lo, uint64_t hi)
{
    u256 r;
    const u128 ll = (u128)lo * lo, lh = (u128)lo * hi, hh = (u128)hi * hi;
    r.w[0] = (uint64_t)ll;
    u128 t = (ll >> 64) + (u128)(uint64_t)lh + (u128)(uint64_t)lh;
    r.w[1] = (uint64_t)t;
    t = (t >> 64) + (lh >> 64) + (lh >> 64) + (u128)(uint64_t)hh;
    r.w[2] = (uint64_t)t;
    t = (t >> 64) + (hh >> 64);
    r.w[3] = (uint64_t)t;
    return r;
}

__device__ __forceinline__ u256 sub_u256(const u256 &a, const u256 &b)
{
    u256 r;
    uint64_t borrow = 0;
    for (int i = 0; i < 4; ++i) {
        const uint64_t d = a.w[i] - b.w[i];
        const uint64_t d2 = d - borrow;
        borrow = (a.w[i] < b.w[i]) || (d < borrow) ? 1u : 0u;
        r.w[i] = d2;
    }
    return r;
}

__device__ __forceinline__ double u256_to_double(const u256 &a)
{
    // top 64 significant bits, rounded once to double, then scaled
    int top = 3;
    while (top > 0 && a.w[top] == 0)
        --top;
    if (top == 0)
        return (double)a.w[0];
    const int lz = __clzll(a.w[top]);
    uint64_t m = lz ? (a.w[top] << lz) | (a.w[top - 1] >> (64 - lz)) : a.w[top];
    // sticky bit for the discarded words
    uint64_t rest = lz ? (a.w[top - 1] << lz) : a.w[top - 1];
    for (int i = top - 2; i >= 0; --i)
        rest |= a.w[i];
    if (rest)
        m |= 1u;
    return ldexp((double)m, 64 * top - lz);
}

__device__ __forceinline__ double u128_div_to_double(uint64_t lo, uint64_t hi,
                                                     uint64_t R)
{
    const u128 v = ((u128)hi << 64) | lo;
    const u128 q = v / R, rem = v % R;
    return (double)q + (double)(uint64_t)rem / (double)R;
}

__global__ __launch_bounds__(256) void micro_moments_kernel(
    uint64_t total, uint64_t R, const uint64_t *__restrict__ sum1,
    const uint64_t *__restrict__ sum2, double *__restrict__ mean,
    double *__restrict__ std_out)
{
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= total)
        return;
    const uint64_t lo = sum1[2 * i], hi = sum1[2 * i + 1];
    mean[i] = u128_div_to_double(lo, hi, R);
    if (R < 2) {
        std_out[i] = __longlong_as_double(0x7FF8000000000000ll); // NaN, as ddof=1
        return;
    }
    const uint64_t s2[3] = {sum2[3 * i], sum2[3 * i + 1], sum2[3 * i + 2]};
    const u256 d = sub_u256(mul_u192_u64(s2, R), square_u128(lo, hi));
    const double num = u256_to_double(d);
    std_out[i] = sqrt(num / ((double)R * (double)(R - 1)));
}

// ---------------------------------------------------------------------------
// Microcanonical statistics with their confidence bounds (the epilogue of
// percolate/percolate.py:557-705) for every step from the exact sums.
// Thread = step s; out[c * S + s] for the 21 columns
//   0..2   max cluster size: mean, lower, upper bound,
//   3..5   spanning: (k + 1) / (R + 2) and the bounds beta[2k], beta[2k + 1]
//          (k = runs with a spanning cluster at s),
//   6 + 3j, 7 + 3j, 8 + 3j   moment j = 0..4: mean, lower, upper bound,
// a bound being mean + (std / sqrt(R)) * t_lo (t_hi) where R > 1 and
// std > 0, the mean otherwise.  Products and sums are rounded one by one
// (no fused multiply-add), as the host's scale * ppf + loc.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void mean_std(const uint64_t *__restrict__ sum1,
                                         const uint64_t *__restrict__ sum2,
                                         uint64_t i, uint64_t R, double &mean,
                                         double &std)
{
    const uint64_t lo = sum1[2 * i], hi = sum1[2 * i + 1];
    mean = u128_div_to_double(lo, hi, R);
    if (R < 2) {
        std = __longlong_as_double(0x7FF8000000000000ll); // NaN, as ddof=1
        return;
    }
    const uint64_t s2[3] = {sum2[3 * i], sum2[3 * i + 1], sum2[3 * i + 2]};
    const u256 d = sub_u256(mul_u192_u64(s2, R), square_u128(lo, hi));
    std = sqrt(u256_to_double(d) / ((double)R * (double)(R - 1)));
}

__global__ __launch_bounds__(256) void micro_ci_kernel(
    uint64_t S, uint64_t R, const uint64_t *__restrict__ sum1,
    const uint64_t *__restrict__ sum2, double t_lo, double t_hi,
    const double *__restrict__ beta, double *__restrict__ out)
{
    // scale * t + mean rounded twice, never fused (HIP contracts by default)
#pragma clang fp contract(off)
    const uint64_t s = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (s >= S)
        return;
    const double sqrt_r = sqrt((double)R);
    // columns of the sums: 0 max, 1 spanning, 2..6 moments 0..4
    const int src[6] = {0, 2, 3, 4, 5, 6};
    const int dst[6] = {0, 6, 9, 12, 15, 18};
    for (int j = 0; j < 6; ++j) {
        double m, sd;
        mean_std(sum1, sum2, (uint64_t)src[j] * S + s, R, m, sd);
        double lo = m, hi = m;
        if (R > 1 && sd != 0.0) {
            const double scale = sd / sqrt_r;
            lo = t_lo * scale + m;
            hi = t_hi * scale + m;
        }
        out[(uint64_t)dst[j] * S + s] = m;
        out[(uint64_t)(dst[j] + 1) * S + s] = lo;
        out[(uint64_t)(dst[j] + 2) * S + s] = hi;
    }
    const uint64_t k = sum1[2 * (S + s)]; // spanning runs (< 2^64)
    out[3 * S + s] = ((double)k + 1.0) / ((double)R + 2.0);
    out[4 * S + s] = beta[2 * k];
    out[5 * S + s] = beta[2 * k + 1];
}

// Finalized canonical averages (percolate/hpc.py:752-834) of P rows of C
// statistics: element i = p * C + c.  Mean and sample standard deviation
// sqrt(M2 / (n - 1)), each divided by div[c] (the number of nodes for the
// per-node statistics, 1 otherwise: x / 1 == x), and the Student-t interval
// q * (std / sqrt(n)) + mean with the caller's per-row quantiles, NaN where
// scipy's ppf refuses its arguments (n - 1 <= 0, scale not > 0, mean NaN).
// out: [4][P][C] = mean, std, lower, upper.
__global__ __launch_bounds__(256) void finalize_kernel(
    uint32_t P, uint32_t C, const uint32_t *__restrict__ runs,
    const double *__restrict__ mean, const double *__restrict__ m2,
    const double *__restrict__ div, const double *__restrict__ q_lo,
    const double *__restrict__ q_hi, double *__restrict__ out)
{
    // every product and sum rounded on its own, as numpy and scipy do
#pragma clang fp contract(off)
    const uint64_t PC = (uint64_t)P * C;
    const uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (i >= PC)
        return;
    const uint32_t p = (uint32_t)(i / C), c = (uint32_t)(i % C);
    const double n = (double)runs[p];
    const double dof = n - 1.0;
    const double d = div[c];
    const double mu = mean[i] / d;
    const double sd = sqrt(m2[i] / dof) / d;
    const double scale = sd / sqrt(n);
    const bool ok = dof > 0.0 && scale > 0.0 && mu == mu;
    const double nan = __longlong_as_double(0x7ff8000000000000ll);
    out[i] = mu;
    out[PC + i] = sd;
    out[2 * PC + i] = ok ? q_lo[p] * scale + mu : nan;
    out[3 * PC + i] = ok ? q_hi[p] * scale + mu : nan;
}

// Pairwise (n, mean, M2) merge of Chan, Golub & LeVeque (the reduction of
// percolate/hpc.py:638-702) of P rows of C statistics: element i = p * C + c,
// per-row counts n_a[p], n_b[p].  mean = mean_a + delta * (n_b / n),
// M2 = M2_a + M2_b + delta^2 * (n_a n_b / n), delta = mean_b - mean_a; the
// outputs may alias the a operands.
__global__ __launch_bounds__(256) void merge_moments_kernel(
    uint64_t PC, uint32_t C, const double *__restrict__ n_a,
    const double *mean_a, const double *m2_a, const double *__restrict__ n_b,
    const double *__restrict__ mean_b, const double *__restrict__ m2_b,
    double *mean_out, double *m2_out)
{
#pragma clang fp contract(off)
    const uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (i >= PC)
        return;
    const uint64_t p = i / C;
    const double na = n_a[p], nb = n_b[p];
    const double n = na + nb;
    const double ma = mean_a[i], delta = mean_b[i] - ma;
    const double m2 = m2_a[i] + m2_b[i] + delta * delta * (na * nb / n);
    mean_out[i] = ma + delta * (nb / n);
    m2_out[i] = m2;
}

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
static const uint32_t kLdsMaxNodes = 16384u;
static const uint32_t kU32RecordMaxNodes = 65536u;
static const uint32_t kSweepMaxNodes = 1u << 28;
static const uint32_t kSumsMaxNodes = 1u << 21;
static const uint32_t kGlobalSlots = 4096u;

static inline hipStream_t as_stream(void *s) { return (hipStream_t)s; }

// parallel merge rounds per batch before the in-order remainder
#ifndef PC_MERGE_ROUNDS
#define PC_MERGE_ROUNDS 4
#endif
static uint32_t g_merge_rounds = PC_MERGE_ROUNDS;

// Two wavefronts per run (a finder and a resolver, see sweep_run) or one:
// unless the caller forces one (PC_SWEEP_ONE_WAVE / PC_SWEEP_TWO_WAVES in
// state_mode), two for HBM state and for LDS state from kSplitMinNodes nodes
// on.  Measured on MI355X: below that the second wave halves the runs a CU
// holds (L = 16: 4.8e10 additions/s with one wave, 3.8e10 with two), above
// it the finder wins (L = 64: 7.0e10 -> 7.4e10; L = 128: 3.3e10 -> 4.1e10).
static const uint32_t kSplitMinNodes = 4096u;

static bool sweep_split(uint32_t num_nodes, bool use_lds, uint32_t waves)
{
    if (waves == PC_SWEEP_ONE_WAVE)
        return false;
    if (waves == PC_SWEEP_TWO_WAVES)
        return true;
    return !use_lds || num_nodes >= kSplitMinNodes;
}

template <bool SPLIT>
static size_t sweep_lds_bytes(uint32_t num_nodes)
{
    return sweep_lds_words<SPLIT>() * sizeof(uint32_t) +
           (((size_t)num_nodes * sizeof(uint16_t) + 3u) & ~(size_t)3u);
}

extern "C" int pc_abi_version(void) { return 1; }

extern "C" const char *pc_last_error(void) { return g_last_error; }

extern "C" int pc_record_bytes(uint32_t num_nodes)
{
    return num_nodes <= kU32RecordMaxNodes ? 4 : 8;
}

// Bucket bits and chunks of the device permutations for num_edges edges.
static void shuffle_plan(uint32_t num_edges, uint32_t &lb1, uint32_t &chunks)
{
    lb1 = 0;
    if (num_edges > SHUF_WHOLE)
        while (((uint64_t)SHUF_BUCKET << lb1) < num_edges)
            ++lb1;
    chunks = (num_edges + SHUF_CHUNK - 1u) / SHUF_CHUNK;
}

extern "C" int pc_permute_philox_workspace_size(uint32_t num_edges,
                                                uint32_t num_runs,
                                                uint64_t *bytes)
{
    g_last_error[0] = 0;
    if (!bytes)
        return pc_fail(PC_EINVAL, "pc_permute_philox_workspace_size: bytes is NULL");
    if (num_edges > SHUF_MAX_EDGES)
        return pc_fail(PC_EOVERFLOW, "pc_permute_philox_workspace_size: num_edges > 2^23");
    uint32_t lb1 = 0, chunks = 0;
    shuffle_plan(num_edges, lb1, chunks);
    const uint64_t nb1 = 1ull << lb1;
    // a run of one bucket is shuffled in LDS from the identity: no counts
    *bytes = lb1 ? (uint64_t)num_runs * (nb1 * chunks + nb1 + 1u) * 4u : 0u;
    return PC_OK;
}

extern "C" int pc_permute_philox_occupancy(uint32_t num_edges, int32_t *blocks_per_cu)
{
    g_last_error[0] = 0;
    if (!blocks_per_cu)
        return pc_fail(PC_EINVAL, "pc_permute_philox_occupancy: NULL output");
    if (num_edges > SHUF_MAX_EDGES)
        return pc_fail(PC_EOVERFLOW, "pc_permute_philox_occupancy: num_edges > 2^23");
    int blocks = 0;
    if (num_edges <= SHUF_SMALL_CAP)
        PC_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &blocks, shuffle_group_kernel<2, true>, 128,
            shuf_group_lds_bytes(2, num_edges, MATCH_BITS)));
    else if (num_edges <= SHUF_WHOLE)
        PC_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &blocks, shuffle_group_kernel<8, true>, 512,
            shuf_group_lds_bytes(8, num_edges, shuf_match_bits(num_edges, 0xFFFFFFFFu))));
    else
        PC_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &blocks, shuffle_group_kernel<4, false>, 256,
            shuf_group_lds_bytes(4, SHUF_GROUP_CAP, MATCH_BITS)));
    *blocks_per_cu = blocks;
    return PC_OK;
}

extern "C" int pc_permute_philox(uint64_t seed, uint64_t first_run,
                                 uint32_t num_runs, uint32_t num_edges,
                                 int32_t *d_perm, int64_t perm_stride,
                                 void *d_workspace, uint64_t workspace_bytes,
                                 void *stream)
{
    g_last_error[0] = 0;
    if (num_runs == 0 || num_edges == 0)
        return PC_OK;
    if (!d_perm || perm_stride < (int64_t)num_edges)
        return pc_fail(PC_EINVAL, "pc_permute_philox: bad output buffer");
    if (num_edges > SHUF_MAX_EDGES)
        return pc_fail(PC_EOVERFLOW, "pc_permute_philox: num_edges > 2^23");
    if (first_run + num_runs > (1ull << 32))
        return pc_fail(PC_EOVERFLOW, "pc_permute_philox: run indices reach 2^32");
    uint64_t need = 0;
    pc_permute_philox_workspace_size(num_edges, num_runs, &need);
    if (need && (!d_workspace || workspace_bytes < need))
        return pc_fail(PC_ENOMEM, "pc_permute_philox: workspace needs %llu bytes",
                       (unsigned long long)need);
    uint32_t lb1 = 0, chunks = 0;
    shuffle_plan(num_edges, lb1, chunks);
    const uint32_t nb1 = 1u << lb1;
    uint32_t *counts = (uint32_t *)d_workspace;
    uint32_t *starts = counts ? counts + (uint64_t)num_runs * nb1 * chunks : nullptr;
    const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
    const uint32_t fr = (uint32_t)first_run;
    hipStream_t s = as_stream(stream);
    // runs in slabs of at most 65535 (the grid's y extent)
    for (uint32_t r0 = 0; r0 < num_runs; r0 += 65535u) {
        const uint32_t rn = min(num_runs - r0, 65535u);
        if (lb1 == 0u && num_edges <= SHUF_SMALL_CAP) {
            shuffle_group_kernel<2, true><<<dim3(1, rn), 128,
                                            shuf_group_lds_bytes(2, num_edges, MATCH_BITS),
                                            s>>>(
                k0, k1, fr, 0u, r0, num_edges, MATCH_BITS, nullptr, d_perm, perm_stride);
            PC_LAUNCH_CHECK("shuffle_group_kernel");
            continue;
        }
        if (lb1 == 0u) {
            const uint32_t in_lds = shuf_match_bits(num_edges, rn);
            shuffle_group_kernel<8, true><<<dim3(1, rn), 512,
                                            shuf_group_lds_bytes(8, num_edges, in_lds), s>>>(
                k0, k1, fr, 0u, r0, num_edges, in_lds, nullptr, d_perm, perm_stride);
            PC_LAUNCH_CHECK("shuffle_group_kernel");
            continue;
        }
        shuffle_count_kernel<<<shuf_blocks(chunks, rn), 64 * SHUF_W, nb1 * 4u, s>>>(
            k0, k1, fr, num_edges, lb1, chunks, r0, rn, counts);
        PC_LAUNCH_CHECK("shuffle_count_kernel");
        shuffle_scan_kernel<<<rn, 256, nb1 * 4u, s>>>(num_edges, lb1, chunks, r0,
                                                      counts, starts);
        PC_LAUNCH_CHECK("shuffle_scan_kernel");
        shuffle_scatter_kernel<<<shuf_blocks(chunks, rn), 64 * SHUF_W,
                                 (SHUF_W + 1u) * nb1 * 4u, s>>>(
            k0, k1, fr, num_edges, lb1, chunks, r0, rn, counts, d_perm, perm_stride);
        PC_LAUNCH_CHECK("shuffle_scatter_kernel");
        shuffle_group_kernel<4, false><<<dim3(nb1, rn), 256,
                                         shuf_group_lds_bytes(4, SHUF_GROUP_CAP, MATCH_BITS),
                                         s>>>(
            k0, k1, fr, lb1, r0, SHUF_GROUP_CAP, MATCH_BITS, starts, d_perm, perm_stride);
        PC_LAUNCH_CHECK("shuffle_group_kernel");
    }
    return PC_OK;
}

extern "C" int pc_sweep_workspace_size(uint32_t num_nodes, uint32_t num_runs,
                                       uint32_t state_mode, uint64_t *bytes)
{
    g_last_error[0] = 0;
    if (!bytes)
        return pc_fail(PC_EINVAL, "pc_sweep_workspace_size: bytes is NULL");
    state_mode &= ~PC_SWEEP_WAVES_MASK;
    if (state_mode == PC_STATE_LDS ||
        (state_mode == PC_STATE_AUTO && num_nodes <= kLdsMaxNodes)) {
        *bytes = 0;
    } else {
        const uint64_t slots = num_runs < kGlobalSlots ? num_runs : kGlobalSlots;
        *bytes = slots * (uint64_t)num_nodes * sizeof(uint32_t);
    }
    return PC_OK;
}

// The sweep launch for either edge source (pc_sweep, pc_sweep_lattice).
template <class ES>
static int sweep_launch(uint32_t num_nodes, uint32_t num_edges, ES edges,
                        bool have_edges, const uint8_t *d_node_sides,
                        int32_t span_on_first_merge, const int32_t *d_perm,
                        int64_t perm_stride, uint32_t num_runs, void *d_records,
                        int64_t rec_stride, uint32_t *d_span_step,
                        void *d_workspace, uint64_t workspace_bytes,
                        uint32_t merge_rounds, uint32_t state_mode,
                        uint64_t *d_chunk_state, void *stream)
{
    const uint32_t rounds = merge_rounds ? merge_rounds : g_merge_rounds;
    if (rounds > 64)
        return pc_fail(PC_EINVAL, "pc_sweep: merge_rounds > 64");
    const uint32_t waves = state_mode & PC_SWEEP_WAVES_MASK;
    state_mode &= ~PC_SWEEP_WAVES_MASK;
    if (state_mode > PC_STATE_HBM || waves == PC_SWEEP_WAVES_MASK)
        return pc_fail(PC_EINVAL, "pc_sweep: unknown state_mode %u", state_mode | waves);
    if (state_mode == PC_STATE_LDS && num_nodes > kLdsMaxNodes)
        return pc_fail(PC_EINVAL, "pc_sweep: LDS state needs num_nodes <= %u",
                       kLdsMaxNodes);
    const bool use_lds = state_mode == PC_STATE_LDS ||
                         (state_mode == PC_STATE_AUTO && num_nodes <= kLdsMaxNodes);
    g_last_error[0] = 0;
    if (num_runs == 0)
        return PC_OK;
    if (num_nodes == 0)
        return pc_fail(PC_EINVAL, "pc_sweep: num_nodes must be positive");
    if (num_nodes > kSweepMaxNodes)
        return pc_fail(PC_EOVERFLOW, "pc_sweep: num_nodes > 2^28");
    if (!d_span_step || (num_edges && (!have_edges || !d_perm || !d_records)))
        return pc_fail(PC_EINVAL, "pc_sweep: NULL buffer");
    if (num_edges && (perm_stride < (int64_t)num_edges ||
                      rec_stride < (int64_t)num_edges))
        return pc_fail(PC_EINVAL, "pc_sweep: stride smaller than num_edges");
    hipStream_t s = as_stream(stream);
    const bool u32rec = num_nodes <= kU32RecordMaxNodes;
    const bool split = sweep_split(num_nodes, use_lds, waves);
    // HBM state with chunk states: a third wave folds the records
    const bool folder = !use_lds && split && d_chunk_state;
    const uint32_t threads = folder ? 192u : split ? 128u : 64u;
    if (use_lds) {
        const size_t lds = split ? sweep_lds_bytes<true>(num_nodes)
                                 : sweep_lds_bytes<false>(num_nodes);
#define PC_SWEEP_LDS(CH, SP, CS)                                                    \
    sweep_lds_kernel<uint32_t, CH, SP, ES><<<num_runs, threads, lds, s>>>(               \
        num_nodes, num_edges, edges, d_node_sides, span_on_first_merge, d_perm,     \
        perm_stride, (uint32_t *)d_records, rec_stride, d_span_step, rounds, CS)
        if (d_chunk_state && split)
            PC_SWEEP_LDS(true, true, d_chunk_state);
        else if (d_chunk_state)
            PC_SWEEP_LDS(true, false, d_chunk_state);
        else if (split)
            PC_SWEEP_LDS(false, true, nullptr);
        else
            PC_SWEEP_LDS(false, false, nullptr);
#undef PC_SWEEP_LDS
        PC_LAUNCH_CHECK("sweep_lds_kernel");
        return PC_OK;
    }
    uint64_t need = 0;
    pc_sweep_workspace_size(num_nodes, num_runs, state_mode, &need);
    if (!d_workspace || workspace_bytes < (uint64_t)num_nodes * 4u)
        return pc_fail(PC_ENOMEM,
                       "pc_sweep: workspace of %llu bytes too small (need %llu)",
                       (unsigned long long)workspace_bytes,
                       (unsigned long long)need);
    uint64_t slots = workspace_bytes / ((uint64_t)num_nodes * 4u);
    if (slots > num_runs)
        slots = num_runs;
    if (slots > kGlobalSlots)
        slots = kGlobalSlots;
#define PC_SWEEP_GLOBAL(RT, CH, SP, FO)                                        \
    sweep_global_kernel<RT, CH, SP, ES, FO><<<(uint32_t)slots, threads, 0, s>>>(   \
        num_nodes, num_edges, num_runs, edges, d_node_sides,                   \
        span_on_first_merge, d_perm, perm_stride, (RT *)d_records, rec_stride, \
        d_span_step, (uint32_t *)d_workspace, rounds, d_chunk_state, nullptr)
#define PC_SWEEP_GLOBAL_W(RT, CH)                                              \
    do {                                                                       \
        if (split)                                                             \
            PC_SWEEP_GLOBAL(RT, CH, true, false);                              \
        else                                                                   \
            PC_SWEEP_GLOBAL(RT, CH, false, false);                             \
    } while (0)
    if (folder && u32rec)
        PC_SWEEP_GLOBAL(uint32_t, true, true, true);
    else if (folder)
        PC_SWEEP_GLOBAL(uint64_t, true, true, true);
    else if (u32rec && d_chunk_state)
        PC_SWEEP_GLOBAL_W(uint32_t, true);
    else if (u32rec)
        PC_SWEEP_GLOBAL_W(uint32_t, false);
    else if (d_chunk_state)
        PC_SWEEP_GLOBAL_W(uint64_t, true);
    else
        PC_SWEEP_GLOBAL_W(uint64_t, false);
#undef PC_SWEEP_GLOBAL_W
#undef PC_SWEEP_GLOBAL
    PC_LAUNCH_CHECK("sweep_global_kernel");
    return PC_OK;
}

extern "C" int pc_sweep(uint32_t num_nodes, uint32_t num_edges,
                        const int32_t *d_edges, const uint8_t *d_node_sides,
                        int32_t span_on_first_merge, const int32_t *d_perm,
                        int64_t perm_stride, uint32_t num_runs, void *d_records,
                        int64_t rec_stride, uint32_t *d_span_step,
                        void *d_workspace, uint64_t workspace_bytes,
                        uint32_t merge_rounds, uint32_t state_mode,
                        uint64_t *d_chunk_state, void *stream)
{
    return sweep_launch(num_nodes, num_edges, EdgeList{(const int2 *)d_edges},
                        d_edges != nullptr, d_node_sides, span_on_first_merge,
                        d_perm, perm_stride, num_runs, d_records, rec_stride,
                        d_span_step, d_workspace, workspace_bytes, merge_rounds,
                        state_mode, d_chunk_state, stream);
}

static LatticeEdges lattice_edges(uint32_t length, bool tiled)
{
    const uint32_t d = 2u * length - 1u;
    return LatticeEdges{length, d, 1.0f / (float)d, tiled ? 1u : 0u};
}

// ---------------------------------------------------------------------------
// The tiled sweep's plan and launches
// ---------------------------------------------------------------------------
// Lattices it takes, and their tiles; false otherwise.
// - A side of at most TILE_MAX_LENGTH, and more than a tile's.
// - Below TILE_LDS_LENGTH (a state that fits LDS several times a CU), batches
//   of at most four runs per CU only.  The sweep in microseconds, untiled and
//   tiled: one run of L = 65 184 and 142, of L = 80 280 and 183, of L = 95 364
//   and 219; 1024 runs 227 and 224, 318 and 292, 422 and 368; 2000 runs 252 and
//   341, 353 and 491, 847 and 657; 8000 runs 896 and 1111, 1432 and 1580, 2426
//   and 2148.  (From L = 88 on the tiles win at 2000 runs and more too, but not
//   at 1500 of L = 95: 473 and 489.)  From TILE_LDS_LENGTH on 2680 and 2360 for
//   8000 of L = 100, 7060 and 5050 for 10^4 of L = 128, 660 and 470 for 200.
// - Tiles of at most 64 x 64 nodes, or 32 x 32 up to L = 128 where those would
//   leave the GPU with at most 2048 wavefronts: more tiles make more events.
//   Sweep in milliseconds with 64 and 32, 200 runs of L = 128 0.479 and 0.412,
//   600 0.547 and 0.548; 500 of L = 100 0.365 and 0.357, 1000 0.445 and 0.491;
//   100 of L = 181 0.598 and 0.597, 200 0.629 and 0.668; 50 of L = 256 0.83 and
//   0.89; 10 of L = 512 2.08 and 2.63.
static bool tile_geo(uint32_t length, bool tiled, uint32_t num_runs, TileGeo &g)
{
    if (length <= TILE_SIDE || length > TILE_MAX_LENGTH ||
        (length < TILE_LDS_LENGTH && num_runs > 1024u))
        return false;
    const uint32_t k64 = (length + TILE_SIDE - 1u) / TILE_SIDE;
    const bool small = length <= 128u && (uint64_t)k64 * k64 * num_runs <= 2048u;
    const uint32_t side = small ? TILE_SIDE / 2u : TILE_SIDE;
    g.lat = lattice_edges(length, tiled);
    g.L = length;
    g.KH = g.KW = (length + side - 1u) / side;
    g.h = g.w = (length + g.KH - 1u) / g.KH;
    g.K = g.KH * g.KW;
    g.per = 2u * g.w + 2u * (g.h - 2u);
    g.mh = (uint32_t)(((1ull << 32) + g.h - 1u) / g.h);
    g.mw = (uint32_t)(((1ull << 32) + g.w - 1u) / g.w);
    g.md = (uint32_t)(((1ull << 32) + g.lat.d - 1u) / g.lat.d);
    g.init_stride = (g.h * g.w + 7u) & ~7u;
    return true;
}

// The workspace of a tiled sweep of num_runs runs whose lists are held for
// `slab` runs at a time: the offsets of its parts, and its size.
struct TilePlan {
    uint64_t init, open, odd, states, counts, windows, lists, list_bytes, bytes;
    uint32_t nodes, slab;
    bool lds;       // the open nodes' codes fit LDS
};
#define TILE_OPEN_LDS_NODES 10240u  // 40 KiB of codes: two runs per CU
#define TILE_OPEN_LDS_MOST 32768u   // 128 KiB: one run per CU

static TilePlan tile_plan(const TileGeo &g, uint32_t num_runs, uint32_t slab)
{
    TilePlan p;
    auto up = [](uint64_t v) { return (v + 255u) & ~(uint64_t)255u; };
    const uint64_t M = 2ull * g.L * (g.L - 1u);
    p.nodes = g.K * g.per;
    p.slab = slab;
    // in LDS also where it holds one run per CU, if the runs are that few
    p.lds = p.nodes <= TILE_OPEN_LDS_NODES ||
            (p.nodes <= TILE_OPEN_LDS_MOST && num_runs <= 256u);
    p.init = 0;
    p.open = up((uint64_t)g.K * g.init_stride * 2u);
    p.odd = p.open + up((uint64_t)p.nodes * 4u);
    p.states = p.odd + up((uint64_t)num_runs * 4u);
    p.counts = p.states + (p.lds ? 0u : up((uint64_t)num_runs * p.nodes * 4u));
    p.windows = p.counts + up(((uint64_t)slab + TILE_SCATTER_BLOCKS) * g.K * 4u);
    p.lists = p.windows + (M > TILE_WINDOW ? up((uint64_t)slab * tile_windows((uint32_t)M) * g.K * 4u) : 0u);
    p.list_bytes = up(M * 4u);
    p.bytes = p.lists + slab * p.list_bytes;
    return p;
}

// Runs whose lists are held at a time: enough (run, tile) wavefronts to fill
// the GPU several times over (16384), more where that takes no more memory
// than the untiled sweep's codes.
static uint32_t tile_slab(const TileGeo &g, uint32_t num_runs)
{
    const uint64_t slots = std::min(num_runs, kGlobalSlots);
    const uint64_t same = slots * g.L * g.L * 4u / tile_plan(g, 1u, 1u).list_bytes;
    const uint64_t fill = (16384u + g.K - 1u) / g.K;
    return (uint32_t)std::min<uint64_t>(num_runs, std::max(same, fill));
}

extern "C" int pc_sweep_lattice_workspace_size(uint32_t length, uint32_t num_runs,
                                               uint32_t state_mode, uint64_t *bytes)
{
    g_last_error[0] = 0;
    if (!bytes)
        return pc_fail(PC_EINVAL, "pc_sweep_lattice_workspace_size: bytes is NULL");
    if (length == 0 || length > 16384u)
        return pc_fail(PC_EINVAL, "pc_sweep_lattice_workspace_size: length must be in 1..16384");
    const int rc = pc_sweep_workspace_size(length * length, num_runs, state_mode, bytes);
    TileGeo g;
    if (rc == PC_OK && num_runs && state_mode == PC_STATE_AUTO &&
        tile_geo(length, false, num_runs, g))
        *bytes = std::max(*bytes, tile_plan(g, num_runs, tile_slab(g, num_runs)).bytes);
    return rc;
}

template <typename RecT>
static int tile_sweep_launch(const TileGeo &g, const TilePlan &p,
                             const uint8_t *d_node_sides, const int32_t *d_perm,
                             int64_t perm_stride, uint32_t num_runs, RecT *d_records,
                             int64_t rec_stride, uint32_t *d_span_step, char *ws,
                             uint32_t rounds, hipStream_t s)
{
    const uint32_t M = 2u * g.L * (g.L - 1u);
    uint16_t *init = (uint16_t *)(ws + p.init);
    uint32_t *open = (uint32_t *)(ws + p.open), *odd = (uint32_t *)(ws + p.odd);
    uint32_t *counts = (uint32_t *)(ws + p.counts);
    uint32_t *windows = (uint32_t *)(ws + p.windows), *lists = (uint32_t *)(ws + p.lists);
    const int64_t list_stride = (int64_t)(p.list_bytes / 4u);
    uint32_t bits = 0;
    while ((1u << bits) < g.K)
        ++bits;
    tile_init_kernel<<<g.K, 256, 0, s>>>(g, d_node_sides, init, open);
    PC_LAUNCH_CHECK("tile_init_kernel");
    for (uint32_t r0 = 0; r0 < num_runs; r0 += p.slab) {
        const uint32_t rn = std::min(p.slab, num_runs - r0);
        const int32_t *perm = d_perm + (int64_t)r0 * perm_stride;
        RecT *rec = d_records + (int64_t)r0 * rec_stride;
        // a workgroup per run, or several where the runs are few: the steps
        // of a segment then start where a count of the earlier ones says
        uint32_t nseg = (TILE_SCATTER_BLOCKS + rn - 1u) / rn;
        nseg = std::min(nseg, (M + 16383u) / 16384u);
        const bool many = g.K > TILE_MANY && M / nseg >= TILE_LONG_SEGMENT;
        // (32-bit records: at most 16 tiles)
        constexpr uint32_t MANY = sizeof(RecT) == 8u ? TILE_GROUPS_MANY : TILE_GROUPS;
        const uint32_t quant = 256u * (many ? MANY : TILE_GROUPS);
        const uint32_t seg = ((M + nseg - 1u) / nseg + quant - 1u) / quant * quant;
        nseg = (M + seg - 1u) / seg;
        if (nseg > 1u) {
            tile_count_kernel<<<dim3(nseg, rn), 256, g.K * 4u, s>>>(g, M, seg, perm,
                                                                    perm_stride, counts);
            PC_LAUNCH_CHECK("tile_count_kernel");
            tile_scan_kernel<<<rn, 256, 0, s>>>(g, nseg, counts, odd + r0);
            PC_LAUNCH_CHECK("tile_scan_kernel");
        }
        auto *scatter = many ? tile_scatter_kernel<RecT, MANY>
                             : tile_scatter_kernel<RecT, TILE_GROUPS>;
        scatter<<<dim3(nseg, rn), 256, 5u * g.K * 4u, s>>>(
            g, M, bits, seg, perm, perm_stride, counts, lists, list_stride, windows, rec,
            rec_stride, d_span_step + r0, odd + r0);
        PC_LAUNCH_CHECK("tile_scatter_kernel");
        const size_t lds = TILE_CLAIM_SLOTS * 4u + g.init_stride * 2u;
        tile_sweep_kernel<RecT><<<shuf_blocks(g.K, rn), 64, lds, s>>>(
            g, rn, lists, list_stride, windows, init, rec, rec_stride, d_span_step + r0,
            odd + r0);
        PC_LAUNCH_CHECK("tile_sweep_kernel");
    }
    const uint32_t threads = 64u * (1u + EVENT_FINDERS);
    if (p.lds)
        event_sweep_kernel<RecT, true><<<num_runs, threads, p.nodes * 4u, s>>>(
            p.nodes, M, open, nullptr, d_records, rec_stride, d_span_step, odd);
    else
        event_sweep_kernel<RecT, false><<<num_runs, threads, 0, s>>>(
            p.nodes, M, open, (uint32_t *)(ws + p.states), d_records, rec_stride,
            d_span_step, odd);
    PC_LAUNCH_CHECK("event_sweep_kernel");
    // runs whose row is not a permutation, with their codes in the lists'
    // place
    const uint64_t slots = p.slab * p.list_bytes / ((uint64_t)g.L * g.L * 4u);
    const uint32_t grid = (uint32_t)std::min<uint64_t>(std::min<uint64_t>(slots, num_runs), 256u);
    sweep_global_kernel<RecT, false, true, LatticeEdges><<<grid, 128, 0, s>>>(
        g.L * g.L, M, num_runs, g.lat, d_node_sides, 0, d_perm, perm_stride, d_records,
        rec_stride, d_span_step, (uint32_t *)lists, rounds, nullptr, odd);
    PC_LAUNCH_CHECK("sweep_global_kernel");
    return PC_OK;
}

// Runs whose lists the tiled sweep of such a call holds at a time, 0 if it
// does not take the call.  Not taken: modes that ask for a state or a number
// of wavefronts, auxiliary sides joined from the first merge on, more than
// 2^31 grid blocks, or a workspace that holds the lists of fewer than 4 runs
// (or of all runs).
static uint32_t tile_runs(uint32_t length, bool tiled, int32_t span_on_first_merge,
                          uint32_t num_runs, uint64_t workspace_bytes,
                          uint32_t state_mode, TileGeo &g)
{
    if (state_mode != PC_STATE_AUTO || span_on_first_merge || num_runs == 0 ||
        !tile_geo(length, tiled, num_runs, g))
        return 0u;
    const uint32_t M = 2u * length * (length - 1u);
    uint32_t slab = tile_slab(g, num_runs);
    if (workspace_bytes < tile_plan(g, num_runs, slab).bytes) {
        const TilePlan one = tile_plan(g, num_runs, 1u);
        const uint64_t per_run = one.list_bytes + (1u + tile_windows(M)) * g.K * 4u;
        const uint64_t base = one.bytes + 512u;
        slab = workspace_bytes < base ? 0u : (uint32_t)std::min<uint64_t>(
                   slab, 1u + (workspace_bytes - base) / per_run);
        if (slab < std::min(num_runs, 4u))
            return 0u;
    }
    // slabs of about the same size, in groups of eight runs
    const uint32_t slabs = (num_runs + slab - 1u) / slab;
    slab = std::min(slab, ((num_runs + slabs - 1u) / slabs + 7u) & ~7u);
    if (slab > 65535u)
        slab = 65528u;
    if (tile_plan(g, num_runs, slab).bytes > workspace_bytes ||
        (uint64_t)(slab + 7u) * g.K > 0x7FFFFFFFu)
        return 0u;
    return slab;
}

extern "C" int pc_sweep_lattice_tiled_runs(uint32_t length, int32_t span_on_first_merge,
                                           uint32_t num_runs, uint64_t workspace_bytes,
                                           uint32_t state_mode, uint32_t *runs)
{
    g_last_error[0] = 0;
    if (!runs)
        return pc_fail(PC_EINVAL, "pc_sweep_lattice_tiled_runs: runs is NULL");
    if (length == 0 || length > 16384u)
        return pc_fail(PC_EINVAL, "pc_sweep_lattice_tiled_runs: length must be in 1..16384");
    TileGeo g;
    *runs = tile_runs(length, false, span_on_first_merge, num_runs, workspace_bytes,
                      state_mode, g);
    return PC_OK;
}

// The tiled sweep, if it takes this call (tile_runs, and a workspace aligned
// for it): *taken tells.
static int tile_sweep(uint32_t length, bool tiled, const uint8_t *d_node_sides,
                      int32_t span_on_first_merge, const int32_t *d_perm,
                      int64_t perm_stride, uint32_t num_runs, void *d_records,
                      int64_t rec_stride, uint32_t *d_span_step, void *d_workspace,
                      uint64_t workspace_bytes, uint32_t merge_rounds,
                      uint32_t state_mode, uint64_t *d_chunk_state, void *stream,
                      bool *taken)
{
    *taken = false;
    TileGeo g;
    const uint32_t rounds = merge_rounds ? merge_rounds : g_merge_rounds;
    const int64_t M = 2ll * length * (length - 1ll);
    if (rounds > 64 || !d_workspace || ((uintptr_t)d_workspace & 15u) || !d_span_step ||
        !d_perm || !d_records || perm_stride < M || rec_stride < M)
        return PC_OK;
    const uint32_t slab = tile_runs(length, tiled, span_on_first_merge, num_runs,
                                    workspace_bytes, state_mode, g);
    if (slab == 0u)
        return PC_OK;
    const TilePlan p = tile_plan(g, num_runs, slab);
    *taken = true;
    hipStream_t s = as_stream(stream);
    const bool u32rec = length * length <= kU32RecordMaxNodes;
    int rc;
    if (u32rec)
        rc = tile_sweep_launch<uint32_t>(
            g, p, d_node_sides, d_perm, perm_stride, num_runs, (uint32_t *)d_records,
            rec_stride, d_span_step, (char *)d_workspace, rounds, s);
    else
        rc = tile_sweep_launch<uint64_t>(
            g, p, d_node_sides, d_perm, perm_stride, num_runs, (uint64_t *)d_records,
            rec_stride, d_span_step, (char *)d_workspace, rounds, s);
    if (rc == PC_OK && d_chunk_state)
        rc = pc_chunk_scan(length * length, (uint32_t)M, num_runs, d_records, rec_stride,
                           d_chunk_state, stream);
    return rc;
}

extern "C" int pc_sweep_lattice(uint32_t length, int32_t tiled,
                                const uint8_t *d_node_sides,
                                int32_t span_on_first_merge, const int32_t *d_perm,
                                int64_t perm_stride, uint32_t num_runs,
                                void *d_records, int64_t rec_stride,
                                uint32_t *d_span_step, void *d_workspace,
                                uint64_t workspace_bytes, uint32_t merge_rounds,
                                uint32_t state_mode, uint64_t *d_chunk_state,
                                void *stream)
{
    g_last_error[0] = 0;
    if (length == 0 || length > 16384u)
        return pc_fail(PC_EINVAL, "pc_sweep_lattice: length must be in 1..16384");
    if (tiled && (length % 8u))
        return pc_fail(PC_EINVAL, "pc_sweep_lattice: the tiled order needs a multiple of 8");
    const uint32_t N = length * length, M = 2u * length * (length - 1u);
    bool taken = false;
    const int rc = tile_sweep(length, tiled != 0, d_node_sides, span_on_first_merge, d_perm,
                              perm_stride, num_runs, d_records, rec_stride, d_span_step,
                              d_workspace, workspace_bytes, merge_rounds, state_mode,
                              d_chunk_state, stream, &taken);
    if (taken)
        return rc;
    return sweep_launch(N, M, lattice_edges(length, tiled != 0), true, d_node_sides,
                        span_on_first_merge, d_perm, perm_stride, num_runs,
                        d_records, rec_stride, d_span_step, d_workspace,
                        workspace_bytes, merge_rounds, state_mode, d_chunk_state,
                        stream);
}

extern "C" int pc_chunk_scan(uint32_t num_nodes, uint32_t num_edges,
                             uint32_t num_runs, const void *d_records,
                             int64_t rec_stride, uint64_t *d_chunk_state,
                             void *stream)
{
    g_last_error[0] = 0;
    if (num_runs == 0 || num_edges == 0)
        return PC_OK;
    if (num_nodes == 0 || num_nodes > kSweepMaxNodes)
        return pc_fail(PC_EOVERFLOW, "pc_chunk_scan: num_nodes out of range");
    if (!d_records || !d_chunk_state || rec_stride < (int64_t)num_edges)
        return pc_fail(PC_EINVAL, "pc_chunk_scan: bad buffer");
    hipStream_t s = as_stream(stream);
    const uint32_t C = (num_edges + 63u) / 64u;
    const uint64_t blocks = (uint64_t)((C + CHUNK_DELTA_PER_BLOCK - 1u) / CHUNK_DELTA_PER_BLOCK) *
                            num_runs;
    if (blocks > 0x7FFFFFFFu)
        return pc_fail(PC_EOVERFLOW, "pc_chunk_scan: too many runs x chunks in one call");
    const dim3 grid((uint32_t)blocks);
    if (num_nodes <= kLdsMaxNodes)
        chunk_delta_kernel<uint32_t, false><<<grid, 64, 0, s>>>(
            num_edges, (const uint32_t *)d_records, rec_stride, d_chunk_state);
    else if (num_nodes <= kU32RecordMaxNodes)
        chunk_delta_kernel<uint32_t, true><<<grid, 64, 0, s>>>(
            num_edges, (const uint32_t *)d_records, rec_stride, d_chunk_state);
    else
        chunk_delta_kernel<uint64_t, true><<<grid, 64, 0, s>>>(
            num_edges, (const uint64_t *)d_records, rec_stride, d_chunk_state);
    PC_LAUNCH_CHECK("chunk_delta_kernel");
    if (num_nodes <= kLdsMaxNodes)
        chunk_prefix_kernel<false><<<num_runs, 64, 0, s>>>(num_nodes, num_edges,
                                                           d_chunk_state);
    else
        chunk_prefix_kernel<true><<<num_runs, 64, 0, s>>>(num_nodes, num_edges,
                                                          d_chunk_state);
    PC_LAUNCH_CHECK("chunk_prefix_kernel");
    return PC_OK;
}

extern "C" int pc_microcanonical_sums(uint32_t num_nodes, uint32_t num_edges,
                                      uint32_t num_runs, const void *d_records,
                                      int64_t rec_stride,
                                      const uint32_t *d_span_step,
                                      const uint64_t *d_chunk_state,
                                      uint64_t *d_sum1, uint64_t *d_sum2,
                                      int32_t accumulate, void *stream)
{
    g_last_error[0] = 0;
    if (num_nodes == 0 || num_nodes > kSumsMaxNodes)
        return pc_fail(PC_EOVERFLOW,
                       "pc_microcanonical_sums: num_nodes outside 1..2^21");
    if (num_nodes <= kLdsMaxNodes) {
        // the 128-bit sums of squares hold R * (N^4 / 8)^2
        const double n4 = (double)num_nodes * num_nodes * num_nodes * num_nodes / 8.0;
        if ((double)num_runs * n4 * n4 >= 0x1p127)
            return pc_fail(PC_EOVERFLOW,
                           "pc_microcanonical_sums: too many runs for N = %u",
                           num_nodes);
    }
    if (!d_sum1 || !d_sum2 || (num_runs && num_edges &&
                               (!d_records || !d_span_step || !d_chunk_state)))
        return pc_fail(PC_EINVAL, "pc_microcanonical_sums: NULL buffer");
    hipStream_t s = as_stream(stream);
    const uint64_t S = (uint64_t)num_edges + 1u;
    const uint32_t C = (num_edges + 63u) / 64u;
    // enough waves to fill 256 CUs several times over, and enough runs a
    // workgroup that its loop outweighs its 29 to 35 atomics a step
    const uint32_t per32 = (num_runs + SUMS_RUNS - 1u) / SUMS_RUNS;
    const bool few = accumulate && (uint64_t)num_runs * C <= (num_runs == 1u ? SUMS_FEW_ONE : SUMS_FEW);
    const bool one_wave = few || (uint64_t)C * per32 >= SUMS_BLOCKS;
    uint32_t groups = C ? (SUMS_BLOCKS / (one_wave ? 1u : 4u) + C - 1u) / C : 1u;
    groups = std::min(groups, few ? num_runs : one_wave ? per32 : (per32 + 1u) / 2u);
    // the bounds of the sums in a group
    groups = std::max(groups, num_runs / SUMS_MOST + (num_runs % SUMS_MOST != 0u));
    const uint32_t rpg = groups ? (num_runs + groups - 1u) / groups : 0u;
    groups = rpg ? (num_runs + rpg - 1u) / rpg : 0u;
    // one group that does not accumulate stores its sums
    const bool store = groups == 1u && !accumulate && num_edges;
    if (!accumulate && !store) {
        fill_zero_kernel<<<1024, 256, 0, s>>>(d_sum1, 7u * S * 2u);
        fill_zero_kernel<<<1024, 256, 0, s>>>(d_sum2, 7u * S * 3u);
        PC_LAUNCH_CHECK("fill_zero_kernel");
    }
    if (num_runs == 0)
        return PC_OK;
    if (num_edges == 0) {
        step0_sums_kernel<<<1, 1, 0, s>>>(num_nodes, num_runs, S, d_sum1, d_sum2);
        PC_LAUNCH_CHECK("step0_sums_kernel");
        return PC_OK;
    }
    const dim3 grid(C, groups);
#define PC_SUMS(RT, WD)                                                               \
    do {                                                                              \
        if (one_wave)                                                                 \
            micro_sums_kernel<RT, WD, 1u><<<grid, 64, 0, s>>>(                        \
                num_nodes, num_edges, num_runs, rpg, (const RT *)d_records,           \
                rec_stride, d_span_step, d_chunk_state, d_sum1, d_sum2, store);       \
        else                                                                          \
            micro_sums_kernel<RT, WD, 4u><<<grid, 256, 0, s>>>(                       \
                num_nodes, num_edges, num_runs, rpg, (const RT *)d_records,           \
                rec_stride, d_span_step, d_chunk_state, d_sum1, d_sum2, store);       \
    } while (0)
    if (num_nodes <= kLdsMaxNodes)
        PC_SUMS(uint32_t, false);
    else if (num_nodes <= kU32RecordMaxNodes)
        PC_SUMS(uint32_t, true);
    else
        PC_SUMS(uint64_t, true);
#undef PC_SUMS
    PC_LAUNCH_CHECK("micro_sums_kernel");
    return PC_OK;
}

extern "C" int pc_expand_traces(uint32_t num_nodes, uint32_t num_edges,
                                uint32_t num_runs, const void *d_records,
                                int64_t rec_stride, const uint32_t *d_span_step,
                                const uint64_t *d_chunk_state,
                                uint32_t *d_max_size, uint8_t *d_spanning,
                                uint64_t *d_moments, void *stream)
{
    g_last_error[0] = 0;
    if (num_runs == 0)
        return PC_OK;
    if (num_nodes == 0 || num_nodes > kSumsMaxNodes)
        return pc_fail(PC_EOVERFLOW, "pc_expand_traces: num_nodes outside 1..2^21");
    if (!d_max_size || !d_spanning || !d_moments ||
        (num_edges && (!d_records || !d_span_step || !d_chunk_state)))
        return pc_fail(PC_EINVAL, "pc_expand_traces: NULL buffer");
    hipStream_t s = as_stream(stream);
    const uint64_t S = (uint64_t)num_edges + 1u;
    if (num_edges == 0) {
        expand_step0_kernel<<<(num_runs + 255u) / 256u, 256, 0, s>>>(
            num_nodes, num_runs, S, d_max_size, d_spanning, d_moments);
        PC_LAUNCH_CHECK("expand_step0_kernel");
        return PC_OK;
    }
    const uint32_t C = (num_edges + 63u) / 64u;
    const dim3 grid(C, num_runs);
    if (num_nodes <= kLdsMaxNodes)
        expand_kernel<uint32_t, false><<<grid, 64, 0, s>>>(
            num_nodes, num_edges, (const uint32_t *)d_records, rec_stride,
            d_span_step, d_chunk_state, d_max_size, d_spanning, d_moments);
    else if (num_nodes <= kU32RecordMaxNodes)
        expand_kernel<uint32_t, true><<<grid, 64, 0, s>>>(
            num_nodes, num_edges, (const uint32_t *)d_records, rec_stride,
            d_span_step, d_chunk_state, d_max_size, d_spanning, d_moments);
    else
        expand_kernel<uint64_t, true><<<grid, 64, 0, s>>>(
            num_nodes, num_edges, (const uint64_t *)d_records, rec_stride,
            d_span_step, d_chunk_state, d_max_size, d_spanning, d_moments);
    PC_LAUNCH_CHECK("expand_kernel");
    return PC_OK;
}

extern "C" int pc_expand_rows(uint32_t num_nodes, uint32_t num_edges, uint32_t num_runs,
                              const int32_t *d_perm, int64_t perm_stride,
                              const void *d_records, int64_t rec_stride,
                              const uint32_t *d_span_step, const uint64_t *d_chunk_state,
                              int32_t spanning, uint8_t *d_rows, void *stream)
{
    g_last_error[0] = 0;
    if (num_runs == 0)
        return PC_OK;
    if (num_nodes == 0 || num_nodes > kSumsMaxNodes)
        return pc_fail(PC_EOVERFLOW, "pc_expand_rows: num_nodes outside 1..2^21");
    if (num_edges == 0 || !d_perm || !d_records || !d_span_step || !d_chunk_state || !d_rows ||
        perm_stride < (int64_t)num_edges || rec_stride < (int64_t)num_edges)
        return pc_fail(PC_EINVAL, "pc_expand_rows: bad buffer");
    hipStream_t s = as_stream(stream);
    const dim3 grid((num_edges + 63u) / 64u, num_runs);
    auto launch = [&](auto rec, auto wide) {
        using RecT = decltype(rec);
        constexpr bool WIDE = decltype(wide)::value;
        auto *kernel = spanning ? expand_rows_kernel<RecT, WIDE, true>
                                : expand_rows_kernel<RecT, WIDE, false>;
        kernel<<<grid, 64, 0, s>>>(num_nodes, num_edges, d_perm, perm_stride,
                                   (const RecT *)d_records, rec_stride, d_span_step,
                                   d_chunk_state, d_rows);
    };
    if (num_nodes <= kLdsMaxNodes)
        launch(uint32_t(), std::false_type());
    else if (num_nodes <= kU32RecordMaxNodes)
        launch(uint32_t(), std::true_type());
    else
        launch(uint64_t(), std::true_type());
    PC_LAUNCH_CHECK("expand_rows_kernel");
    return PC_OK;
}

extern "C" int pc_binomial_window(uint32_t n, double p, int64_t *start,
                                  int64_t *len)
{
    g_last_error[0] = 0;
    if (!start || !len)
        return pc_fail(PC_EINVAL, "pc_binomial_window: NULL output");
    if (!(p >= 0.0 && p <= 1.0))
        return pc_fail(PC_EINVAL, "pc_binomial_window: p outside [0, 1]");
    const double mu = (double)n * p;
    const double sigma = sqrt((double)n * p * (1.0 - p));
    const double half = 12.0 * sigma + 48.0;
    double lo = floor(mu - half), hi = ceil(mu + half);
    if (lo < 0.0)
        lo = 0.0;
    if (hi > (double)n)
        hi = (double)n;
    *start = (int64_t)lo;
    *len = (int64_t)hi - (int64_t)lo + 1;
    return PC_OK;
}

// The p of a launch travel in its arguments (480 fit beside the pointers in
// the 4 KB that a launch may carry): no copy, and no wait for one.  A call of
// pc_canonical_fused with its grid (L = 128, 201 p, 21 columns) took 229 us
// with the windows found on the host and four copies, 33 us with this.
#define GRID_PS 480u
struct GridPs {
    double p[GRID_PS];
};

__global__ __launch_bounds__(GRID_PS) void binomial_grid_kernel(
    GridPs g, uint32_t count, uint32_t n, double *__restrict__ ps,
    int64_t *__restrict__ start, int64_t *__restrict__ len)
{
#pragma clang fp contract(off)
    const uint32_t i = threadIdx.x;
    if (i >= count)
        return;
    // pc_binomial_window, operation for operation
    const double p = g.p[i];
    const double mu = (double)n * p;
    const double sigma = __dsqrt_rn((double)n * p * (1.0 - p));
    const double half = 12.0 * sigma + 48.0;
    const double lo = max(floor(mu - half), 0.0), hi = min(ceil(mu + half), (double)n);
    ps[i] = p;
    start[i] = (int64_t)lo;
    len[i] = (int64_t)hi - (int64_t)lo + 1;
}

extern "C" int pc_binomial_grid(uint32_t n, uint32_t num_p, const double *ps, double *d_ps,
                                int64_t *d_start, int64_t *d_len, void *stream)
{
    g_last_error[0] = 0;
    if (num_p == 0)
        return PC_OK;
    if (!ps || !d_ps || !d_start || !d_len)
        return pc_fail(PC_EINVAL, "pc_binomial_grid: NULL buffer");
    for (uint32_t i = 0; i < num_p; ++i)
        if (!(ps[i] >= 0.0 && ps[i] <= 1.0))
            return pc_fail(PC_EINVAL, "pc_binomial_grid: p outside [0, 1]");
    hipStream_t s = as_stream(stream);
    for (uint32_t i = 0; i < num_p; i += GRID_PS) {
        GridPs g;
        const uint32_t count = std::min(GRID_PS, num_p - i);
        memcpy(g.p, ps + i, count * sizeof(double));
        binomial_grid_kernel<<<1, GRID_PS, 0, s>>>(g, count, n, d_ps + i, d_start + i, d_len + i);
        PC_LAUNCH_CHECK("binomial_grid_kernel");
    }
    return PC_OK;
}

extern "C" int pc_binomial_weights(uint32_t n, uint32_t num_p,
                                   const double *d_ps, const int64_t *d_start,
                                   const int64_t *d_len, int64_t kmax,
                                   double *d_w, void *stream)
{
    g_last_error[0] = 0;
    if (num_p == 0)
        return PC_OK;
    if (!d_ps || !d_start || !d_len || !d_w || kmax <= 0)
        return pc_fail(PC_EINVAL, "pc_binomial_weights: bad buffer");
    hipStream_t s = as_stream(stream);
    const dim3 grid((uint32_t)((kmax + 255) / 256), num_p);
    binom_weights_kernel<<<grid, 256, 0, s>>>(n, d_ps, d_start, d_len, kmax, d_w);
    PC_LAUNCH_CHECK("binom_weights_kernel");
    binom_normalize_kernel<<<num_p, 256, 0, s>>>(kmax, d_len, d_w);
    PC_LAUNCH_CHECK("binom_normalize_kernel");
    return PC_OK;
}

// K-slices of the MFMA contraction: enough tiles x slices to fill the GPU
// with about 16k wavefronts, at most PC_CONTRACT_SLICES.
#ifndef PC_CONTRACT_WAVES
#define PC_CONTRACT_WAVES 16384u
#endif
static uint32_t contract_slices(uint32_t num_p, uint32_t cols)
{
    const uint64_t tiles = (uint64_t)((num_p + 15u) / 16u) * ((cols + 15u) / 16u);
    uint64_t sl = (PC_CONTRACT_WAVES + tiles - 1u) / (tiles ? tiles : 1u);
    if (sl < 1u)
        sl = 1u;
    if (sl > PC_CONTRACT_SLICES)
        sl = PC_CONTRACT_SLICES;
    return (uint32_t)sl;
}

// The FP64 matrix-core contraction takes the wide kernel from this many
// columns on, with tiles of 64 p x WIDE_TC columns.
#define WIDE_TC 64
#define WIDE_MIN_COLS WIDE_TC

static bool contract_wide(uint32_t cols, int32_t precision)
{
    return precision == PC_PREC_FP64_MFMA && cols >= (uint32_t)WIDE_MIN_COLS;
}

static uint32_t wide_tiles_p(uint32_t num_p) { return (num_p + WIDE_TILE - 1u) / WIDE_TILE; }
static uint32_t wide_tiles(uint32_t num_p, uint32_t cols)
{
    return wide_tiles_p(num_p) * ((cols + WIDE_TC - 1u) / WIDE_TC);
}

// K-slices of the wide kernel: none from four workgroups per CU on (1024
// tiles), otherwise enough to reach about that many, at most 16.
static uint32_t wide_slices(uint32_t num_p, uint32_t cols)
{
    const uint64_t tiles = wide_tiles(num_p, cols);
    if (tiles >= 1024u)
        return 1u;
    uint64_t sl = (1024u + tiles - 1u) / (tiles ? tiles : 1u);
    return (uint32_t)(sl > PC_CONTRACT_SLICES ? PC_CONTRACT_SLICES : sl);
}

extern "C" int pc_contract_workspace_size(uint32_t num_p, uint32_t cols,
                                          int32_t precision, uint64_t *bytes)
{
    g_last_error[0] = 0;
    if (!bytes)
        return pc_fail(PC_EINVAL, "pc_contract_workspace_size: bytes is NULL");
    if (precision == PC_PREC_FP64)
        *bytes = 0u;
    else if (contract_wide(cols, precision)) {
        const uint32_t sl = wide_slices(num_p, cols);
        *bytes = sl > 1u ? (uint64_t)sl * num_p * cols * sizeof(double) : 0u;
    } else
        *bytes = (uint64_t)contract_slices(num_p, cols) * num_p * cols *
                 sizeof(double);
    return PC_OK;
}

extern "C" int pc_canonical_contract(uint32_t num_steps, uint32_t cols,
                                     const void *d_x, int64_t x_stride,
                                     uint32_t num_p, const int64_t *d_start,
                                     const int64_t *d_len, const void *d_w,
                                     int64_t kmax, double *d_out,
                                     int32_t precision, void *d_workspace,
                                     uint64_t workspace_bytes, void *stream)
{
    g_last_error[0] = 0;
    if (num_p == 0 || cols == 0)
        return PC_OK;
    if (precision == PC_PREC_FP64 && cols > CONTRACT_MAX_COLS)
        return pc_fail(PC_EOVERFLOW,
                       "pc_canonical_contract: FP64 vector form takes at most %d columns",
                       CONTRACT_MAX_COLS);
    if (!d_x || !d_start || !d_len || !d_w || !d_out || x_stride < (int64_t)cols)
        return pc_fail(PC_EINVAL, "pc_canonical_contract: bad buffer");
    hipStream_t s = as_stream(stream);
    if (precision == PC_PREC_FP64) {
        const double *x = (const double *)d_x, *w = (const double *)d_w;
        if (cols <= 8)
            contract_f64_kernel<8><<<num_p, 256, 0, s>>>(
                x, num_steps, x_stride, d_start, d_len, w, kmax, d_out, (int32_t)cols);
        else if (cols <= 16)
            contract_f64_kernel<16><<<num_p, 256, 0, s>>>(
                x, num_steps, x_stride, d_start, d_len, w, kmax, d_out, (int32_t)cols);
        else
            contract_f64_kernel<32><<<num_p, 256, 0, s>>>(
                x, num_steps, x_stride, d_start, d_len, w, kmax, d_out, (int32_t)cols);
        PC_LAUNCH_CHECK("contract_f64_kernel");
        return PC_OK;
    }
    uint64_t need = 0;
    pc_contract_workspace_size(num_p, cols, precision, &need);
    if (need > 0u && (!d_workspace || workspace_bytes < need))
        return pc_fail(PC_ENOMEM, "pc_canonical_contract: workspace needs %llu bytes",
                       (unsigned long long)need);
    const TileCtx t{num_p, cols, x_stride, kmax, d_start, d_len};
    if (contract_wide(cols, precision)) {
        const uint32_t sl = wide_slices(num_p, cols);
        const dim3 grid(wide_tiles(num_p, cols), sl);
        double *dst = sl > 1u ? (double *)d_workspace : d_out;
        contract_wide_f64_kernel<WIDE_TC><<<grid, 256, 0, s>>>(
            (const double *)d_x, num_steps, (const double *)d_w, t,
            wide_tiles_p(num_p), sl, dst);
        PC_LAUNCH_CHECK("contract_wide_f64_kernel");
        if (sl > 1u) {
            const int64_t n = (int64_t)num_p * cols;
            contract_reduce_kernel<<<(uint32_t)((n + 255) / 256), 256, 0, s>>>(
                dst, sl, n, d_out);
            PC_LAUNCH_CHECK("contract_reduce_kernel");
        }
        return PC_OK;
    }
    const uint32_t slices = contract_slices(num_p, cols);
    const dim3 grid((num_p + 15u) / 16u, (cols + 15u) / 16u, slices);
    double *partial = (double *)d_workspace;
    switch (precision) {
    case PC_PREC_FP64_MFMA:
        contract_mfma_kernel<PC_PREC_FP64_MFMA><<<grid, 64, 0, s>>>(
            d_x, num_steps, d_w, t, slices, partial);
        break;
    case PC_PREC_FP32_MFMA:
        contract_mfma_kernel<PC_PREC_FP32_MFMA><<<grid, 64, 0, s>>>(
            d_x, num_steps, d_w, t, slices, partial);
        break;
    case PC_PREC_BF16X3_MFMA:
        contract_mfma_kernel<PC_PREC_BF16X3_MFMA><<<grid, 64, 0, s>>>(
            d_x, num_steps, d_w, t, slices, partial);
        break;
    default:
        return pc_fail(PC_EINVAL, "pc_canonical_contract: unknown precision %d",
                       precision);
    }
    PC_LAUNCH_CHECK("contract_mfma_kernel");
    const int64_t n = (int64_t)num_p * cols;
    contract_reduce_kernel<<<(uint32_t)((n + 255) / 256), 256, 0, s>>>(
        partial, slices, n, d_out);
    PC_LAUNCH_CHECK("contract_reduce_kernel");
    return PC_OK;
}

extern "C" int pc_canonical_fused_workspace_size(uint32_t num_p, uint32_t cols,
                                                 int32_t precision, uint64_t *bytes)
{
    g_last_error[0] = 0;
    if (!bytes)
        return pc_fail(PC_EINVAL, "pc_canonical_fused_workspace_size: bytes is NULL");
    if (precision != PC_PREC_FP64_MFMA && precision != PC_PREC_SPLIT_BF16)
        return pc_fail(PC_EINVAL, "pc_canonical_fused_workspace_size: unknown precision %d",
                       precision);
    *bytes = (uint64_t)contract_slices(num_p, cols + 1u) * num_p * (cols + 1u) *
             sizeof(double);
    return PC_OK;
}

// Checks of pc_canonical_fused's arguments; returns PC_OK or a failure.
static int fused_check(const char *who, uint32_t cols, const double *d_x,
                       int64_t x_stride, const double *d_ps,
                       const int64_t *d_start, const int64_t *d_len,
                       double *d_out)
{
    if (cols > 4096u)
        return pc_fail(PC_EOVERFLOW, "%s: at most 4096 columns", who);
    if (!d_x || !d_ps || !d_start || !d_len || !d_out || x_stride < (int64_t)cols)
        return pc_fail(PC_EINVAL, "%s: bad buffer", who);
    return PC_OK;
}

// The launches of pc_canonical_fused with the partial sums in `partial`
// (pc_canonical_fused_workspace_size bytes; every entry is written before
// it is read, so it needs no clearing).
static int fused_launch(uint32_t num_edges, uint32_t cols, const double *d_x,
                        int64_t x_stride, uint32_t num_p, const double *d_ps,
                        const int64_t *d_start, const int64_t *d_len,
                        double *d_out, int32_t precision, double *partial,
                        hipStream_t s)
{
    const FusedCtx f{d_x, x_stride, d_ps, d_start, d_len, num_edges, num_p, cols};
    const uint32_t slices = contract_slices(num_p, cols + 1u);
    const dim3 grid((num_p + 15u) / 16u, (cols + 1u + 15u) / 16u, slices);
    if (precision == PC_PREC_FP64_MFMA) {
        canonical_fused_f64_kernel<<<grid, 64, 0, s>>>(f, slices, partial);
        PC_LAUNCH_CHECK("canonical_fused_f64_kernel");
    } else {
        canonical_fused_split_kernel<<<grid, 64, 0, s>>>(f, slices, partial);
        PC_LAUNCH_CHECK("canonical_fused_split_kernel");
    }
    const int64_t n = (int64_t)num_p * cols;
    fused_reduce_kernel<<<(uint32_t)((n + 255) / 256), 256, 0, s>>>(
        partial, slices, num_p, cols, d_out);
    PC_LAUNCH_CHECK("fused_reduce_kernel");
    return PC_OK;
}

extern "C" int pc_canonical_fused(uint32_t num_edges, uint32_t cols,
                                  const double *d_x, int64_t x_stride,
                                  uint32_t num_p, const double *d_ps,
                                  const int64_t *d_start, const int64_t *d_len,
                                  double *d_out, int32_t precision,
                                  void *d_workspace, uint64_t workspace_bytes,
                                  void *stream)
{
    g_last_error[0] = 0;
    if (num_p == 0 || cols == 0)
        return PC_OK;
    int rc = fused_check("pc_canonical_fused", cols, d_x, x_stride, d_ps,
                         d_start, d_len, d_out);
    if (rc != PC_OK)
        return rc;
    uint64_t need = 0;
    if (pc_canonical_fused_workspace_size(num_p, cols, precision, &need) != PC_OK)
        return PC_EINVAL;
    if (!d_workspace || workspace_bytes < need)
        return pc_fail(PC_ENOMEM, "pc_canonical_fused: workspace needs %llu bytes",
                       (unsigned long long)need);
    return fused_launch(num_edges, cols, d_x, x_stride, num_p, d_ps, d_start,
                        d_len, d_out, precision, (double *)d_workspace,
                        as_stream(stream));
}

// ---------------------------------------------------------------------------
// Scratch of pc_canonical_fused_noalloc: a file-scope device array, one copy
// per GPU, held until the process ends.  Host code never passes the array's
// name to a kernel (on the host it is only a stand-in for the symbol): the
// device address of each GPU's copy comes from hipGetSymbolAddress, looked
// up once per device with that device current, and is used everywhere.
// ---------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[PC_NOALLOC_SCRATCH_BYTES];

#define PC_MAX_DEVICES 64
static std::mutex g_scratch_mutex;
static void *g_scratch_ptr[PC_MAX_DEVICES];

// Device address of the current device's scratch copy.
static int scratch_address(void **out)
{
    int dev = -1;
    PC_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= PC_MAX_DEVICES)
        return pc_fail(PC_EINVAL, "scratch: device ordinal %d outside 0..%d", dev,
                       PC_MAX_DEVICES - 1);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        PC_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p)
            return pc_fail(PC_EHIP, "scratch: hipGetSymbolAddress gave NULL");
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return PC_OK;
}

extern "C" int pc_canonical_fused_noalloc(uint32_t num_edges, uint32_t cols,
                                          const double *d_x, int64_t x_stride,
                                          uint32_t num_p, const double *d_ps,
                                          const int64_t *d_start,
                                          const int64_t *d_len, double *d_out,
                                          int32_t precision, void *stream)
{
    g_last_error[0] = 0;
    if (num_p == 0 || cols == 0)
        return PC_OK;
    int rc = fused_check("pc_canonical_fused_noalloc", cols, d_x, x_stride, d_ps,
                         d_start, d_len, d_out);
    if (rc != PC_OK)
        return rc;
    uint64_t need = 0;
    if (pc_canonical_fused_workspace_size(num_p, cols, precision, &need) != PC_OK)
        return PC_EINVAL;
    if (need > (uint64_t)PC_NOALLOC_SCRATCH_BYTES)
        return pc_fail(PC_ENOMEM,
                       "pc_canonical_fused_noalloc: %u p x %u columns need %llu "
                       "bytes of scratch, above the fixed %u (use "
                       "pc_canonical_fused with a workspace)",
                       num_p, cols, (unsigned long long)need,
                       (unsigned)PC_NOALLOC_SCRATCH_BYTES);
    void *p = nullptr;
    rc = scratch_address(&p);
    if (rc != PC_OK)
        return rc;
    return fused_launch(num_edges, cols, d_x, x_stride, num_p, d_ps, d_start,
                        d_len, d_out, precision, (double *)p, as_stream(stream));
}

extern "C" int pc_convert_f64_to_f32(const double *d_in, int64_t n, float *d_out,
                                     void *stream)
{
    g_last_error[0] = 0;
    if (n <= 0)
        return PC_OK;
    if (!d_in || !d_out)
        return pc_fail(PC_EINVAL, "pc_convert_f64_to_f32: NULL buffer");
    f64_to_f32_kernel<<<2048, 256, 0, as_stream(stream)>>>(d_in, n, d_out);
    PC_LAUNCH_CHECK("f64_to_f32_kernel");
    return PC_OK;
}

extern "C" int pc_microcanonical_ci(uint32_t num_edges, uint32_t num_runs,
                                    const uint64_t *d_sum1, const uint64_t *d_sum2,
                                    double t_lo, double t_hi, const double *d_beta,
                                    double *d_out, void *stream)
{
    g_last_error[0] = 0;
    if (num_runs == 0)
        return pc_fail(PC_EINVAL, "pc_microcanonical_ci: no runs");
    if (!d_sum1 || !d_sum2 || !d_beta || !d_out)
        return pc_fail(PC_EINVAL, "pc_microcanonical_ci: NULL buffer");
    const uint64_t S = (uint64_t)num_edges + 1u;
    micro_ci_kernel<<<(uint32_t)((S + 255) / 256), 256, 0, as_stream(stream)>>>(
        S, num_runs, d_sum1, d_sum2, t_lo, t_hi, d_beta, d_out);
    PC_LAUNCH_CHECK("micro_ci_kernel");
    return PC_OK;
}

extern "C" int pc_finalize_canonical(uint32_t num_ps, uint32_t num_columns,
                                     const uint32_t *d_runs, const double *d_mean,
                                     const double *d_m2, const double *d_div,
                                     const double *d_q_lo, const double *d_q_hi,
                                     double *d_out, void *stream)
{
    g_last_error[0] = 0;
    const uint64_t total = (uint64_t)num_ps * num_columns;
    if (total == 0)
        return PC_OK;
    if (!d_runs || !d_mean || !d_m2 || !d_div || !d_q_lo || !d_q_hi || !d_out)
        return pc_fail(PC_EINVAL, "pc_finalize_canonical: NULL buffer");
    if ((total + 255u) / 256u > 0x7FFFFFFFull)
        return pc_fail(PC_EOVERFLOW, "pc_finalize_canonical: too many rows");
    finalize_kernel<<<(uint32_t)((total + 255u) / 256u), 256, 0, as_stream(stream)>>>(
        num_ps, num_columns, d_runs, d_mean, d_m2, d_div, d_q_lo, d_q_hi, d_out);
    PC_LAUNCH_CHECK("finalize_kernel");
    return PC_OK;
}

extern "C" int pc_merge_moments(uint32_t num_ps, uint32_t num_columns,
                                const double *d_n_a, const double *d_mean_a,
                                const double *d_m2_a, const double *d_n_b,
                                const double *d_mean_b, const double *d_m2_b,
                                double *d_mean_out, double *d_m2_out, void *stream)
{
    g_last_error[0] = 0;
    const uint64_t total = (uint64_t)num_ps * num_columns;
    if (total == 0)
        return PC_OK;
    if (!d_n_a || !d_mean_a || !d_m2_a || !d_n_b || !d_mean_b || !d_m2_b ||
        !d_mean_out || !d_m2_out)
        return pc_fail(PC_EINVAL, "pc_merge_moments: NULL buffer");
    if ((total + 255u) / 256u > 0x7FFFFFFFull)
        return pc_fail(PC_EOVERFLOW, "pc_merge_moments: too many rows");
    merge_moments_kernel<<<(uint32_t)((total + 255u) / 256u), 256, 0, as_stream(stream)>>>(
        total, num_columns, d_n_a, d_mean_a, d_m2_a, d_n_b, d_mean_b, d_m2_b,
        d_mean_out, d_m2_out);
    PC_LAUNCH_CHECK("merge_moments_kernel");
    return PC_OK;
}

extern "C" int pc_microcanonical_moments(uint32_t num_edges, uint32_t num_runs,
                                         const uint64_t *d_sum1,
                                         const uint64_t *d_sum2, double *d_mean,
                                         double *d_std, void *stream)
{
    g_last_error[0] = 0;
    if (num_runs == 0)
        return pc_fail(PC_EINVAL, "pc_microcanonical_moments: no runs");
    if (!d_sum1 || !d_sum2 || !d_mean || !d_std)
        return pc_fail(PC_EINVAL, "pc_microcanonical_moments: NULL buffer");
    const uint64_t total = (uint64_t)PC_COLUMNS * ((uint64_t)num_edges + 1u);
    micro_moments_kernel<<<(uint32_t)((total + 255) / 256), 256, 0,
                           as_stream(stream)>>>(total, num_runs, d_sum1, d_sum2,
                                                d_mean, d_std);
    PC_LAUNCH_CHECK("micro_moments_kernel");
    return PC_OK;
}

// Plan of a persistent multi-graph sweep: device table entries, the LDS
// bytes (the largest LDS-state graph), the HBM slot size (the largest
// HBM-state graph), the queue length and the grid (workgroups resident at
// once).
struct MultiPlan {
    std::vector<MultiGraph> table;
    size_t lds;
    uint64_t slot_words, total;
    uint32_t grid;
};

static int multi_plan(uint32_t num_graphs, const pc_sweep_graph *graphs,
                      MultiPlan &plan)
{
    if (num_graphs == 0 || !graphs)
        return pc_fail(PC_EINVAL, "pc_sweep_multi: no graphs");
    plan.table.assign(num_graphs, MultiGraph{});
    plan.lds = sweep_lds_words<true>() * sizeof(uint32_t);
    plan.slot_words = 0;
    plan.total = 0;
    for (uint32_t g = 0; g < num_graphs; ++g) {
        const pc_sweep_graph &in = graphs[g];
        MultiGraph &G = plan.table[g];
        const uint32_t rounds = in.merge_rounds ? in.merge_rounds : g_merge_rounds;
        if (in.num_nodes == 0 || in.num_nodes > kSweepMaxNodes || rounds > 64)
            return pc_fail(PC_EINVAL, "pc_sweep_multi: graph %u: bad sizes", g);
        const uint32_t L = in.lattice_length;
        if (L && ((uint64_t)L * L != in.num_nodes ||
                  in.num_edges != 2u * L * (L - 1u) ||
                  (in.num_nodes > kLdsMaxNodes && (L % 8u))))
            return pc_fail(PC_EINVAL, "pc_sweep_multi: graph %u is not the lattice of "
                           "side %u (tiled order needs a multiple of 8)", g, L);
        if (in.num_runs && in.num_edges &&
            ((!L && !in.d_edges) || !in.d_perm || !in.d_records || !in.d_span_step ||
             !in.d_chunk_state || in.perm_stride < (int64_t)in.num_edges ||
             in.rec_stride < (int64_t)in.num_edges))
            return pc_fail(PC_EINVAL, "pc_sweep_multi: graph %u: bad buffers", g);
        if (in.num_runs && !in.d_span_step)
            return pc_fail(PC_EINVAL, "pc_sweep_multi: graph %u: no span output", g);
        G.edges = (const int2 *)in.d_edges;
        G.lattice = L ? lattice_edges(L, in.num_nodes > kLdsMaxNodes)
                      : LatticeEdges{0u, 1u, 1.0f, 0u};
        G.sides = in.d_node_sides;
        G.perm = in.d_perm;
        G.records = in.d_records;
        G.span_step = in.d_span_step;
        G.chunk_state = in.d_chunk_state;
        G.perm_stride = in.perm_stride;
        G.rec_stride = in.rec_stride;
        G.N = in.num_nodes;
        G.M = in.num_edges;
        G.runs = in.num_runs;
        G.first = (uint32_t)plan.total;
        G.span_first = in.span_on_first_merge ? 1u : 0u;
        G.rounds = rounds;
        G.shift = in.num_nodes > 1u ? 32u - (uint32_t)__builtin_clz(in.num_nodes - 1u) : 0u;
        if (in.num_nodes <= kLdsMaxNodes) {
            G.kind = MULTI_LDS;
            plan.lds = std::max(plan.lds, sweep_lds_bytes<true>(in.num_nodes));
        } else {
            G.kind = in.num_nodes <= kU32RecordMaxNodes ? MULTI_HBM32 : MULTI_HBM64;
            plan.slot_words = std::max<uint64_t>(plan.slot_words, in.num_nodes);
            plan.lds = std::max(plan.lds, (sweep_lds_words<true>() + DIRTY_SLOTS) *
                                              sizeof(uint32_t));
        }
        plan.total += in.num_runs;
    }
    if (plan.total >= (1ull << 32) - 65536u)
        return pc_fail(PC_EOVERFLOW, "pc_sweep_multi: too many runs");
    int dev = 0, cus = 0, blocks = 0;
    PC_HIP_CHECK(hipGetDevice(&dev));
    PC_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    PC_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &blocks, sweep_multi_kernel, 128, plan.lds));
    if (blocks < 1)
        return pc_fail(PC_EINVAL, "pc_sweep_multi: %zu bytes of LDS do not fit", plan.lds);
    uint64_t grid = (uint64_t)cus * (uint64_t)blocks;
    if (grid > plan.total)
        grid = plan.total ? plan.total : 1u;
    plan.grid = (uint32_t)grid;
    return PC_OK;
}

// The table, then the queue head at the next 256-byte boundary.
static uint64_t multi_head_offset(uint32_t num_graphs)
{
    return ((uint64_t)num_graphs * sizeof(MultiGraph) + 255u) & ~(uint64_t)255u;
}
static uint64_t multi_table_bytes(uint32_t num_graphs)
{
    return multi_head_offset(num_graphs) + 256u;
}

extern "C" int pc_sweep_multi_workspace_size(uint32_t num_graphs,
                                             const pc_sweep_graph *graphs,
                                             uint64_t *table_bytes,
                                             uint64_t *workspace_bytes)
{
    g_last_error[0] = 0;
    if (!table_bytes || !workspace_bytes)
        return pc_fail(PC_EINVAL, "pc_sweep_multi_workspace_size: NULL output");
    MultiPlan plan;
    const int rc = multi_plan(num_graphs, graphs, plan);
    if (rc)
        return rc;
    *table_bytes = multi_table_bytes(num_graphs);
    *workspace_bytes = (uint64_t)plan.grid * plan.slot_words * 4u;
    return PC_OK;
}

extern "C" int pc_sweep_multi_prepare(uint32_t num_graphs,
                                      const pc_sweep_graph *graphs,
                                      void *d_table, uint64_t table_bytes)
{
    g_last_error[0] = 0;
    MultiPlan plan;
    const int rc = multi_plan(num_graphs, graphs, plan);
    if (rc)
        return rc;
    const size_t bytes = (size_t)num_graphs * sizeof(MultiGraph);
    if (!d_table || table_bytes < multi_table_bytes(num_graphs) ||
        ((uintptr_t)d_table & 255u))
        return pc_fail(PC_ENOMEM, "pc_sweep_multi_prepare: table needs %llu bytes, "
                       "256-byte aligned",
                       (unsigned long long)multi_table_bytes(num_graphs));
    PC_HIP_CHECK(hipMemcpy(d_table, plan.table.data(), bytes, hipMemcpyHostToDevice));
    return PC_OK;
}

extern "C" int pc_sweep_multi(uint32_t num_graphs, const pc_sweep_graph *graphs,
                              void *d_table, uint64_t table_bytes,
                              void *d_workspace, uint64_t workspace_bytes,
                              void *stream)
{
    g_last_error[0] = 0;
    MultiPlan plan;
    const int rc = multi_plan(num_graphs, graphs, plan);
    if (rc)
        return rc;
    if (!d_table || table_bytes < multi_table_bytes(num_graphs) ||
        ((uintptr_t)d_table & 255u))
        return pc_fail(PC_EINVAL, "pc_sweep_multi: table of %llu bytes too small "
                       "or not 256-byte aligned", (unsigned long long)table_bytes);
    const uint64_t need = (uint64_t)plan.grid * plan.slot_words * 4u;
    if (need && (!d_workspace || workspace_bytes < need))
        return pc_fail(PC_ENOMEM, "pc_sweep_multi: workspace needs %llu bytes",
                       (unsigned long long)need);
    if (plan.total == 0)
        return PC_OK;
    uint32_t *head = (uint32_t *)((char *)d_table + multi_head_offset(num_graphs));
    hipStream_t s = as_stream(stream);
    zero_u32_kernel<<<1, 1, 0, s>>>(head);
    PC_LAUNCH_CHECK("zero_u32_kernel");
    sweep_multi_kernel<<<plan.grid, 128, plan.lds, s>>>(
        (const MultiGraph *)d_table, num_graphs, (uint32_t)plan.total, head,
        (uint32_t *)d_workspace, plan.slot_words);
    PC_LAUNCH_CHECK("sweep_multi_kernel");
    return PC_OK;
}

extern "C" int pc_sweep_occupancy(uint32_t num_nodes, uint32_t state_mode,
                                  int32_t *blocks_per_cu)
{
    g_last_error[0] = 0;
    if (!blocks_per_cu)
        return pc_fail(PC_EINVAL, "pc_sweep_occupancy: NULL output");
    const uint32_t waves = state_mode & PC_SWEEP_WAVES_MASK;
    state_mode &= ~PC_SWEEP_WAVES_MASK;
    if (state_mode > PC_STATE_HBM || waves == PC_SWEEP_WAVES_MASK)
        return pc_fail(PC_EINVAL, "pc_sweep_occupancy: unknown state_mode %u",
                       state_mode | waves);
    int blocks = 0;
    const bool use_lds = state_mode == PC_STATE_LDS ||
                         (state_mode == PC_STATE_AUTO && num_nodes <= kLdsMaxNodes);
    const bool split = sweep_split(num_nodes, use_lds, waves);
    if (use_lds) {
        if (num_nodes > kLdsMaxNodes)
            return pc_fail(PC_EINVAL, "pc_sweep_occupancy: too many nodes for LDS");
        if (split)
            PC_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &blocks, sweep_lds_kernel<uint32_t, false, true, EdgeList>, 128,
                sweep_lds_bytes<true>(num_nodes)));
        else
            PC_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &blocks, sweep_lds_kernel<uint32_t, false, false, EdgeList>, 64,
                sweep_lds_bytes<false>(num_nodes)));
    } else if (split) {
        PC_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &blocks, sweep_global_kernel<uint32_t, false, true, EdgeList>, 128, 0));
    } else {
        PC_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &blocks, sweep_global_kernel<uint32_t, false, false, EdgeList>, 64, 0));
    }
    *blocks_per_cu = blocks;
    return PC_OK;
}

extern "C" int pc_window_traces(uint32_t num_nodes, uint32_t num_edges,
                                uint32_t num_runs, const void *d_records,
                                int64_t rec_stride, const uint32_t *d_span_step,
                                const uint64_t *d_chunk_state, int64_t g_lo,
                                int64_t g_len, int32_t spanning, double *d_out,
                                void *stream)
{
    g_last_error[0] = 0;
    if (num_runs == 0 || g_len <= 0)
        return PC_OK;
    if (num_nodes == 0 || num_nodes > kSumsMaxNodes)
        return pc_fail(PC_EOVERFLOW, "pc_window_traces: num_nodes outside 1..2^21");
    if (g_lo < 0 || g_lo + g_len > (int64_t)num_edges + 1)
        return pc_fail(PC_EINVAL, "pc_window_traces: window outside 0..num_edges");
    if (num_edges == 0)
        return pc_fail(PC_EINVAL, "pc_window_traces: graph without edges");
    if (!d_records || !d_span_step || !d_chunk_state || !d_out)
        return pc_fail(PC_EINVAL, "pc_window_traces: NULL buffer");
    const int64_t first_chunk = g_lo > 0 ? (g_lo - 1) / 64 : 0;
    const int64_t last_step = g_lo + g_len - 1;
    const int64_t last_chunk = last_step > 0 ? (last_step - 1) / 64 : 0;
    const dim3 grid((uint32_t)(last_chunk - first_chunk + 1),
                    (num_runs + WT_RUNS - 1u) / WT_RUNS);
    hipStream_t s = as_stream(stream);
    if (num_nodes <= kLdsMaxNodes)
        window_traces_kernel<uint32_t, false><<<grid, 64, 0, s>>>(
            num_nodes, num_edges, num_runs, (const uint32_t *)d_records,
            rec_stride, d_span_step, d_chunk_state, g_lo, g_len, spanning, d_out);
    else if (num_nodes <= kU32RecordMaxNodes)
        window_traces_kernel<uint32_t, true><<<grid, 64, 0, s>>>(
            num_nodes, num_edges, num_runs, (const uint32_t *)d_records,
            rec_stride, d_span_step, d_chunk_state, g_lo, g_len, spanning, d_out);
    else
        window_traces_kernel<uint64_t, true><<<grid, 64, 0, s>>>(
            num_nodes, num_edges, num_runs, (const uint64_t *)d_records,
            rec_stride, d_span_step, d_chunk_state, g_lo, g_len, spanning, d_out);
    PC_LAUNCH_CHECK("window_traces_kernel");
    return PC_OK;
}

extern "C" int pc_run_moments(const double *d_q, uint32_t num_p,
                              uint32_t num_runs, uint32_t cols, double *d_mean,
                              double *d_m2, void *stream)
{
    g_last_error[0] = 0;
    if (num_p == 0 || cols == 0)
        return PC_OK;
    if (num_runs == 0 || !d_q || !d_mean || !d_m2)
        return pc_fail(PC_EINVAL, "pc_run_moments: bad arguments");
    if (cols > RUN_MOMENTS_COLS)
        return pc_fail(PC_EINVAL, "pc_run_moments: at most 8 columns");
    run_moments_kernel<<<num_p, 256, 0, as_stream(stream)>>>(
        d_q, num_p, num_runs, cols, d_mean, d_m2);
    PC_LAUNCH_CHECK("run_moments_kernel");
    return PC_OK;
}

// Targets of every run: a workgroup each while two fit every CU (200 runs of
// 130560 edges: 0.47 ms, with a wavefront each 0.98; 600 of 79600: 0.70 and
// 0.68).
static int rs_targets(const uint32_t *d_seeds, uint32_t num_runs, uint32_t num_edges,
                      int32_t *d_perm, int64_t perm_stride, hipStream_t s)
{
    if (num_runs <= 512u)
        randomstate_targets_wide_kernel<<<num_runs, RST_T, 0, s>>>(d_seeds, num_edges, d_perm,
                                                                   perm_stride);
    else
        randomstate_targets_kernel<<<num_runs, 64, 0, s>>>(d_seeds, num_edges, d_perm,
                                                           perm_stride);
    PC_LAUNCH_CHECK("randomstate_targets_kernel");
    return PC_OK;
}

extern "C" int pc_permute_randomstate(const uint32_t *d_seeds, uint32_t num_runs,
                                      uint32_t num_edges, int32_t *d_perm,
                                      int64_t perm_stride, void *stream)
{
    g_last_error[0] = 0;
    if (num_runs == 0 || num_edges == 0)
        return PC_OK;
    if (!d_seeds || !d_perm || perm_stride < (int64_t)num_edges)
        return pc_fail(PC_EINVAL, "pc_permute_randomstate: bad buffer");
    if (num_edges > 0x7fffffffu)
        return pc_fail(PC_EOVERFLOW, "pc_permute_randomstate: num_edges >= 2^31");
    hipStream_t s = as_stream(stream);
    if (num_edges <= RS_APPLY_MAX) {
        // targets, then all swaps at once (in place in the output rows)
        const int rc = rs_targets(d_seeds, num_runs, num_edges, d_perm, perm_stride, s);
        if (rc != PC_OK)
            return rc;
        const size_t lds = rs_apply_lds_bytes(num_edges);
        // as few threads and indices per thread as hold the run: 480 edges
        // take 27 us with the largest form
        if (num_edges <= 512u)
            randomstate_apply_kernel<256u, 2u><<<num_runs, 256, lds, s>>>(num_edges, d_perm,
                                                                          perm_stride);
        else if (num_edges <= 4096u)
            randomstate_apply_kernel<512u, 8u><<<num_runs, 512, lds, s>>>(num_edges, d_perm,
                                                                          perm_stride);
        else if (num_edges <= 8192u)
            randomstate_apply_kernel<1024u, 8u><<<num_runs, 1024, lds, s>>>(num_edges, d_perm,
                                                                            perm_stride);
        else
            randomstate_apply_kernel<1024u, 32u><<<num_runs, 1024, lds, s>>>(num_edges, d_perm,
                                                                             perm_stride);
        PC_LAUNCH_CHECK("randomstate_apply_kernel");
        return PC_OK;
    }
    if (num_edges <= MT_LDS_MAX) {
        const size_t lds = ((size_t)num_edges * sizeof(uint16_t) + 3u) & ~(size_t)3u;
        permute_randomstate_kernel<true><<<num_runs, 64, lds, s>>>(
            d_seeds, num_edges, d_perm, perm_stride);
    } else {
        permute_randomstate_kernel<false><<<num_runs, 64, 0, s>>>(
            d_seeds, num_edges, d_perm, perm_stride);
    }
    PC_LAUNCH_CHECK("permute_randomstate_kernel");
    return PC_OK;
}

// Slots of the bucketed second phase, and its workspace: the table, then
// per slot the entries and the values.
#define RSB_SLOTS 512u
static uint64_t rsb_entry_bytes(uint32_t n) { return n <= RSB_SHORT ? 4u : 8u; }
static bool rsb_takes(uint32_t n) { return n > RS_APPLY_MAX && n <= RSB_MAX; }

extern "C" int pc_permute_randomstate_workspace_size(uint32_t num_edges, uint32_t num_runs,
                                                     uint64_t *bytes)
{
    g_last_error[0] = 0;
    if (!bytes)
        return pc_fail(PC_EINVAL, "pc_permute_randomstate_workspace_size: bytes is NULL");
    const uint64_t slots = std::min(num_runs, RSB_SLOTS);
    *bytes = slots && rsb_takes(num_edges)
                 ? sizeof(RsbTable) + 512u + slots * num_edges * (4u + rsb_entry_bytes(num_edges))
                 : 0u;
    return PC_OK;
}

extern "C" int pc_permute_randomstate_ws(const uint32_t *d_seeds, uint32_t num_runs,
                                         uint32_t num_edges, int32_t *d_perm,
                                         int64_t perm_stride, void *d_workspace,
                                         uint64_t workspace_bytes, void *stream)
{
    g_last_error[0] = 0;
    if (num_runs == 0 || num_edges == 0)
        return PC_OK;
    if (!d_seeds || !d_perm || perm_stride < (int64_t)num_edges)
        return pc_fail(PC_EINVAL, "pc_permute_randomstate_ws: bad buffer");
    const uint64_t eb = rsb_entry_bytes(num_edges), per_slot = num_edges * (4u + eb);
    const uint64_t fixed = (sizeof(RsbTable) + 511u) & ~(uint64_t)255u;
    // without room for a run the swaps are walked in sequence
    if (!rsb_takes(num_edges) || !d_workspace || ((uintptr_t)d_workspace & 7u) ||
        workspace_bytes < fixed + per_slot)
        return pc_permute_randomstate(d_seeds, num_runs, num_edges, d_perm, perm_stride, stream);
    const uint32_t slots = (uint32_t)std::min<uint64_t>(
        std::min(num_runs, RSB_SLOTS), (workspace_bytes - fixed) / per_slot);
    uint32_t shift = 0;
    while (((num_edges - 1u) >> shift) >= RSB_CELLS)
        ++shift;
    RsbTable *table = (RsbTable *)d_workspace;
    char *entries = (char *)d_workspace + fixed;
    uint32_t *values = (uint32_t *)(entries + slots * num_edges * eb);
    hipStream_t s = as_stream(stream);
    randomstate_table_kernel<<<32, 256, 0, s>>>(num_edges, shift, table);
    PC_LAUNCH_CHECK("randomstate_table_kernel");
    const int rc = rs_targets(d_seeds, num_runs, num_edges, d_perm, perm_stride, s);
    if (rc != PC_OK)
        return rc;
    if (eb == 4u)
        randomstate_buckets_kernel<uint32_t><<<slots, RSB_T, 0, s>>>(
            num_edges, num_runs, shift, table, (uint32_t *)entries, values, d_perm, perm_stride);
    else
        randomstate_buckets_kernel<uint64_t><<<slots, RSB_T, 0, s>>>(
            num_edges, num_runs, shift, table, (uint64_t *)entries, values, d_perm, perm_stride);
    PC_LAUNCH_CHECK("randomstate_buckets_kernel");
    return PC_OK;
}
