// grt_window.h -- the windowed wave traversal: a wave walks its rays a window
// of cells at a time and spreads the triangle tests of the whole window over
// its 64 lanes.
//
// Per window, every lane steps its ray over a few cells, issuing
// the cells' list bounds together (a DDA does not depend on what the cells
// hold), so the window costs one memory latency instead of one per cell.  The
// lists of all lanes are then laid end to end -- lane by lane, cell by cell --
// and tested 64 or 128 records at a time, whichever ray a record belongs to:
// a wave needs sum / 64 rounds of tests where a per-lane loop needs, cell by
// cell, the maximum over its lanes.  Cells after the one that ends a ray are
// tested in vain; a window is short enough that this costs less than it saves.
//
// The result is the serial one.  Each ray keeps the minimum of an LDS key
// (cell in the window, t, position in the cell's list): the first cell that
// holds a hit decides, inside it the smallest t, among equal t the earliest
// record (the serial loop replaces only on a strictly smaller t).  Any hit
// keeps (cell, position).  Counters count what the serial loop would visit.
#pragma once

#include "grt_mt.h"

namespace grt {

constexpr int kWinCells = 4;         // cells per lane and window, at most
constexpr uint32_t kWinSegs = 64 * kWinCells;
// Lists of at least this many records are tested by the whole wave one at a
// time (64 records a round, the ray in registers), the others pooled.  A long
// list alone fills rounds without the pooled round's bookkeeping: the stadium
// one-level primary stage took 2.39 ms with 1000 here, 2.08 with 192, 2.23
// with 64 (rounds left part empty).  It also bounds the pooled tests of a
// window, so their numbering fits 32 bits for any list length.
constexpr uint32_t kWinLong = 192;

// LDS of one wave.
struct WaveWin {
    float4 ro[64], rd[64];             // each lane's ray: {origin, lo}, {direction, tmin}
    unsigned long long win[64];        // per lane: minimum key
    uint2 seg_rb[kWinSegs];            // {first record - start, end of its hits}
    uint32_t seg_start[kWinSegs];      // first pooled test of the list
    uint32_t mark[128];
    uint16_t seg_own[kWinSegs];        // lane | cell << 6 | second record array << 10
};
static_assert(sizeof(WaveWin) % 16 == 0, "WaveWin arrays stay 16-byte aligned");

// Inclusive prefix maximum over a full wave64 (see wave_incl_scan).
__device__ __forceinline__ uint32_t wave_incl_max(uint32_t v)
{
    const auto mx = [](uint32_t a, uint32_t b) { return a > b ? a : b; };
    v = mx(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true));
    v = mx(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true));
    v = mx(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true));
    v = mx(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true));
    v = mx(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));
    v = mx(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));
    return v;
}

// Order-preserving bits of t, -0 folded into +0.
__device__ __forceinline__ uint32_t win_t_bits(float t)
{
    const uint32_t b = __float_as_uint(t == 0.0f ? 0.0f : t);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

// Keys: cell (4 bits), t (32), position in the list (28).  A built grid lists
// each of a scene's at most 2^28 triangles once per cell; an uploaded one may
// repeat them, so a closest-hit position is modulo kWinSpan: a longer list is
// tested span by span (SPANS), and the one-level walk finds the record again.
// An any-hit key has no t: its position takes those bits too, for any length.
__device__ __forceinline__ unsigned long long win_key(uint32_t cell, uint32_t tbits, uint32_t j)
{
    return ((unsigned long long)cell << 60) | ((unsigned long long)tbits << 28) | j;
}

__device__ __forceinline__ uint32_t win_cell(unsigned long long key)
{
    return (uint32_t)(key >> 60);
}

__device__ __forceinline__ uint32_t win_t_bits(unsigned long long key)
{
    return (uint32_t)(key >> 28);
}

template <bool ANY>
__device__ __forceinline__ uint32_t win_pos(unsigned long long key)
{
    return ANY ? (uint32_t)key : (uint32_t)key & (kWinSpan - 1u);
}

// A ray as the pooled tests read it: {origin, lo} and {direction, tmin}, lo a
// lower bound factor of the filter below.  Its upper end, the smaller of tmax
// and the cell's exit bound, comes with the list.
//
// The filter of mt_maybe without branches (64 unrelated tests take every
// branch): hi * |det| and lo * |det| bound the numerator of t.  hi is at least
// 2^-20, so its product with a guarded |det| does not underflow; lo is 0 for
// tmin 0 (a numerator of 0 or less is a miss), tmin (1 - 2^-19) in the range
// mt_maybe tests, else -inf (no lower bound).  NaN ends never hit.
__device__ __forceinline__ float win_lo(float tmin)
{
    if (tmin == 0.0f)
        return 0.0f;
    return tmin >= 0x1p-20f && tmin <= 0x1p20f ? tmin * (1.0f - 0x1p-19f) : -INFINITY;
}

// The upper end of a list's hits: t <= end exactly when t <= tmax and t <=
// bound (NaN, which no t is at most, when either is NaN).
__device__ __forceinline__ float win_end(float tmax, float bound)
{
    return __builtin_elementwise_minimum(tmax, bound);
}

// Lanes per ray for a wave that holds `rays` rays to walk: `lanes`, doubled
// while the idle lanes allow it, up to `most`.  Shadow and bounce launches
// leave many waves with a few rays; the longest of those end the launch
// (stadium frame 3707 -> 3562 us, 24 served requests 6680 -> 6555, batch of 16
// scenes 552 -> 540; launches of full waves unchanged).
__device__ __forceinline__ uint32_t win_lanes(uint32_t rays, uint32_t lanes, uint32_t most)
{
    while (lanes < most && 2u * lanes * rays <= 64u)
        lanes *= 2u;
    return lanes;
}

// The wave's rays i (heads: the lanes that hold one to walk) regrouped with
// `lanes` lanes per ray, in order: the ray of the calling lane's group, false
// when there is none.
__device__ __forceinline__ bool win_regroup(WaveWin& W, uint64_t heads, uint32_t lanes,
                                            uint32_t& i)
{
    const uint32_t lane = threadIdx.x & 63u;
    if ((heads >> lane) & 1u)
        W.mark[lanes_below(heads)] = i;
    wave_lds_sync();
    const uint32_t g = lane >> __builtin_ctz(lanes);
    const bool valid = g < (uint32_t)__popcll(heads);
    i = W.mark[valid ? g : 0u];
    wave_lds_sync();
    return valid;
}

// One record against one ray; tbits receives the key's t part.
template <bool ANY>
__device__ __forceinline__ bool win_test(const float4 A, const float4 B, const float4 C,
                                         const float4 ro, const float4 rd, float end,
                                         uint32_t& tbits)
{
    const MtPre m = mt_pre(A, B, C, ro.x, ro.y, ro.z, rd.x, rd.y, rd.z);
    const float ad = fabsf(m.det);
    const uint32_t sgn = __float_as_uint(m.det) & 0x80000000u;
    const float us = __uint_as_float(__float_as_uint(m.un) ^ sgn);
    const float vs = __uint_as_float(__float_as_uint(m.vn) ^ sgn);
    const float ts = __uint_as_float(__float_as_uint(m.tn) ^ sgn);
    const float hi = (end > 0x1p-20f ? end : 0x1p-20f) * (1.0f + 0x1p-19f);
    const bool miss = (us < ad * -0x1p-40f) | (vs < ad * -0x1p-40f) |
                      (us + vs > ad * (1.0f + 0x1p-16f)) | (ts > hi * ad) |
                      (ts <= ro.w * ad);
    if (miss & (ad >= 0x1p-100f) & (ad <= 0x1p100f))
        return false;
    float t, u, v;
    if (!(mt_exact(m, t, u, v) && t > rd.w && t <= end))
        return false;
    tbits = ANY ? 0u : win_t_bits(t);
    return ANY || t < INFINITY;
}

// The record arrays that a window's lists point into: a two-level walk mixes
// lists of top cells and of sub-cells.
struct WinRecs {
    const float4* __restrict__ top;
    const float4* __restrict__ sub;
};

// Pooled tests [base, min(base + 64 K, end)), K consecutive ones per lane.
// seg: lists staged, those before k0 start before base; carry: 1 + the list
// holding the test before base.
template <bool ANY, bool TWO, int K>
__device__ __forceinline__ void win_round(WaveWin& W, const WinRecs recs, uint32_t base,
                                          uint32_t end, uint32_t nseg, uint32_t& k0,
                                          uint32_t& carry)
{
    const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
    for (int q = 0; q < K; ++q)
        W.mark[K * lane + q] = 0u;
    wave_lds_sync();
    const uint32_t lim = base + 64u * K;
    uint32_t started = 0;
#pragma unroll
    for (int q = 0; q < K; ++q) {
        const uint32_t k = k0 + 64u * q + lane;
        const uint32_t st = k < nseg ? W.seg_start[k] : 0xffffffffu;
        const bool in = st < lim;
        if (in)
            W.mark[st - base] = k + 1u;
        started += (uint32_t)__popcll(__ballot(in));
    }
    k0 += started;
    wave_lds_sync();
    uint32_t mk[K], top = 0;
#pragma unroll
    for (int q = 0; q < K; ++q) {
        mk[q] = W.mark[K * lane + q];
        top = mk[q] > top ? mk[q] : top;
    }
    const uint32_t incl = wave_incl_max(top);
    uint32_t cur = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x138, 0xf, 0xf, false);
    cur = cur > carry ? cur : carry;
    const uint32_t last = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    carry = last > carry ? last : carry;
    float4 A[K], B[K], C[K];
    uint32_t seg[K], own[K];
    float hit_end[K];
#pragma unroll
    for (int q = 0; q < K; ++q) {
        cur = mk[q] > cur ? mk[q] : cur;
        seg[q] = cur - 1u;
        const uint32_t p = base + K * lane + q;
        const uint2 rb = W.seg_rb[seg[q]];
        const uint64_t ref = (uint32_t)(rb.x + (p < end ? p : end - 1u));
        own[q] = W.seg_own[seg[q]];
        const float4* __restrict__ rec = TWO && (own[q] & 1024u) ? recs.sub : recs.top;
        A[q] = rec[3ull * ref];
        B[q] = rec[3ull * ref + 1];
        C[q] = rec[3ull * ref + 2];
        hit_end[q] = __uint_as_float(rb.y);
    }
#pragma unroll
    for (int q = 0; q < K; ++q) {
        const uint32_t p = base + K * lane + q;
        const uint32_t o = own[q] & 63u;
        const float4 ro = W.ro[o], rd = W.rd[o];
        uint32_t tb;
        if (p < end && win_test<ANY>(A[q], B[q], C[q], ro, rd, hit_end[q], tb))
            atomicMin(&W.win[o], win_key((own[q] >> 6) & 15u, tb, p - W.seg_start[seg[q]]));
    }
}

// Per-cell values of a window: vectors, which stay in registers also where
// they are indexed at run time (arrays went to scratch memory).
template <int S>
using WinU = uint32_t __attribute__((ext_vector_type(S)));

template <int S>
__device__ __forceinline__ uint32_t win_pick(const WinU<S> a, uint32_t s)
{
    uint32_t r = a[0];
#pragma unroll
    for (int q = 1; q < S; ++q)
        r = s == (uint32_t)q ? uint32_t(a[q]) : uint32_t(r);
    return r;
}

__device__ __forceinline__ unsigned long long win_wave_min(unsigned long long v)
{
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long w = __shfl_xor(v, o, 64);
        v = w < v ? w : v;
    }
    return v;
}

// One long list of lane l's ray (cell s of its window): the whole wave, 128
// records a round (n is at most kRefsMax: j0 does not wrap).
template <bool ANY, bool SPANS>
__device__ __forceinline__ void win_long(WaveWin& W, const float4* __restrict__ trir, uint32_t l,
                                         uint32_t s, uint32_t b, uint32_t n, float end)
{
    const uint32_t lane = threadIdx.x & 63u;
    const float4 ro = W.ro[l], rd = W.rd[l];
    unsigned long long key = ~0ull;
    for (uint32_t j0 = 0; j0 < n; j0 += 128u) {
        const uint32_t ja = j0 + lane, jb = ja + 64u;
        const uint64_t ka = b + (ja < n ? ja : n - 1u), kb = b + (jb < n ? jb : n - 1u);
        const float4 A0 = trir[3ull * ka], B0 = trir[3ull * ka + 1], C0 = trir[3ull * ka + 2];
        const float4 A1 = trir[3ull * kb], B1 = trir[3ull * kb + 1], C1 = trir[3ull * kb + 2];
        uint32_t tb;
        if (ja < n && win_test<ANY>(A0, B0, C0, ro, rd, end, tb)) {
            const unsigned long long k = win_key(s, tb, ja);
            key = k < key ? k : key;
        }
        if (jb < n && win_test<ANY>(A1, B1, C1, ro, rd, end, tb)) {
            const unsigned long long k = win_key(s, tb, jb);
            key = k < key ? k : key;
        }
        if (ANY && __ballot(key != ~0ull) != 0)
            break;
    }
    key = win_wave_min(key);
    // at the same t a hit of an earlier span of the list stays
    if (lane == 0 && (SPANS ? (key >> 28) < (W.win[l] >> 28) : key < W.win[l]))
        W.win[l] = key;
}

// All tests of the wave's window: the lane's cells, numbers cell0.. of its
// ray's window, hold the lists [b, b + n) (n = 0: none).  Every lane of the
// wave calls it; W.ro and W.rd hold the rays.  The lanes that share a ray name
// the same owner lane.  Bit s of `subs`: list s is in the second record array
// (TWO).  Returns the ray's key, ~0 without a hit.
template <bool ANY, bool TWO, int S, bool SPANS>
__device__ __forceinline__ unsigned long long win_tests(WaveWin& W, const WinRecs recs,
                                                        const WinU<S> b, const WinU<S> n,
                                                        const WinU<S> end, uint32_t subs,
                                                        uint32_t owner, uint32_t cell0)
{
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t lists = 0, tests = 0, longm = 0;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const bool lng = n[s] >= kWinLong;
        longm |= lng ? 1u << s : 0u;
        lists += (n[s] != 0 && !lng) ? 1u : 0u;
        tests += lng ? 0u : n[s];
    }
    // lists <= 64 S < 2^10 and tests < 64 S kWinLong < 2^22: one scan
    static_assert(S <= kWinCells && kWinSegs < 1024u && kWinSegs * kWinLong < (1u << 22),
                  "packed scan");
    const uint32_t own = (tests << 10) | lists;
    const uint32_t incl = wave_incl_scan(own);
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    const uint32_t all_lists = total & 1023u, all_tests = total >> 10;
    const uint64_t any_long = __ballot(longm != 0);
    if (all_lists == 0 && any_long == 0)
        return ~0ull;
    W.win[lane] = ~0ull;
    wave_lds_sync();
    uint32_t k = (incl - own) & 1023u, st = (incl - own) >> 10;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if (n[s] != 0 && n[s] < kWinLong) {
            W.seg_start[k] = st;
            W.seg_rb[k] = make_uint2(b[s] - st, end[s]);
            W.seg_own[k] = (uint16_t)(owner | ((cell0 + (uint32_t)s) << 6) |
                                      (TWO ? ((subs >> s) & 1u) << 10 : 0u));
            ++k;
            st += n[s];
        }
    }
    wave_lds_sync();
    uint32_t k0 = 0, carry = 0, base = 0;
    for (; base + 64u < all_tests; base += 128u)
        win_round<ANY, TWO, 2>(W, recs, base, all_tests, all_lists, k0, carry);
    if (base < all_tests)
        win_round<ANY, TWO, 1>(W, recs, base, all_tests, all_lists, k0, carry);
    wave_lds_sync();
    if (any_long != 0) {
        uint32_t done = 0;   // records of the list in spans tested already
        for (;;) {
            const uint64_t m = __ballot(longm != 0);
            if (m == 0)
                break;
            const uint32_t l = (uint32_t)__builtin_ctzll(m);
            const uint32_t s = longm != 0 ? (uint32_t)__builtin_ctz(longm) : 0u;
            // an earlier cell of the ray with a hit decides it
            const bool skip = win_cell(W.win[owner]) < cell0 + s;
            const uint32_t lb = win_pick<S>(b, s), ln = win_pick<S>(n, s);
            const uint32_t le = win_pick<S>(end, s);
            const float4* __restrict__ rec =
                TWO && __builtin_amdgcn_readlane((int)((subs >> s) & 1u), (int)l) != 0 ? recs.sub
                                                                                       : recs.top;
            // the span of the list to test now: from record `at` on
            const uint32_t at = done;
            bool rest = true;
            if (SPANS) {
                rest = (uint32_t)__builtin_amdgcn_readlane((int)ln, (int)l) - at <= kWinSpan;
                done = rest ? 0u : at + kWinSpan;
            }
            if (lane == l && rest)
                longm &= longm - 1u;
            if (__builtin_amdgcn_readlane((int)skip, (int)l))
                continue;
            const uint32_t ray = (uint32_t)__builtin_amdgcn_readlane((int)owner, (int)l);
            const uint32_t cell = (uint32_t)__builtin_amdgcn_readlane((int)(cell0 + s), (int)l);
            const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)lb, (int)l) + at;
            const uint32_t left = (uint32_t)__builtin_amdgcn_readlane((int)ln, (int)l) - at;
            win_long<ANY, SPANS>(W, rec, ray, cell, first, rest ? left : kWinSpan,
                                 __int_as_float(__builtin_amdgcn_readlane((int)le, (int)l)));
            wave_lds_sync();
        }
    }
    wave_lds_sync();
    return W.win[owner];
}

}  // namespace grt
