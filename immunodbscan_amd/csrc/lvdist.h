// lvdist.h — "is the Levenshtein distance of x and y at most t" for small t,
// shared by the device kernels and a host-side test (compiled without HIP).
//
// The diagonal method of E. Ukkonen ("Algorithms for approximate string
// matching", Inf. Control 1985; also G. Landau and U. Vishkin, 1989):
// f(e, d) is the furthest position i of x reached on diagonal d (position
// i + d of y) with e edits,
//   f(e, d) = slide_d(max(f(e-1, d) + 1, f(e-1, d-1), f(e-1, d+1) + 1)),
// where slide_d moves on over matching letters; the distance is at most t
// exactly when f(t, ly - lx) reaches the end of x.  Rows are bit planes (bit i
// of plane p = bit p of letter i's code), so the mismatches of a whole
// diagonal are one shift, XOR and OR per plane and word, and a slide is a
// search for the next set bit: no per-letter loop and no per-row tables.
// Positions past min(lx, ly - d) are cut off after the search, so the bits
// beyond a row's end do not matter.
#pragma once
#include <stdint.h>

#ifndef IDB_HD
#if defined(__HIPCC__)
#define IDB_HD __host__ __device__ __forceinline__
#else
#define IDB_HD static inline
#endif
#endif

// ((hi:lo) >> s), 0 <= s <= 31
IDB_HD uint32_t idb_funnel(uint32_t hi, uint32_t lo, uint32_t s)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_alignbit(hi, lo, s);
#else
    return (uint32_t)((((uint64_t)hi << 32) | lo) >> s);
#endif
}

// Index of the lowest set bit, all ones without one.
IDB_HD uint32_t idb_low_bit(uint32_t v) { return v ? (uint32_t)__builtin_ctz(v) : 0xFFFFFFFFu; }

IDB_HD uint32_t idb_reverse(uint32_t v)
{
#if defined(__clang__)
    return __builtin_bitreverse32(v);
#else
    v = ((v >> 1) & 0x55555555u) | ((v & 0x55555555u) << 1);
    v = ((v >> 2) & 0x33333333u) | ((v & 0x33333333u) << 2);
    v = ((v >> 4) & 0x0F0F0F0Fu) | ((v & 0x0F0F0F0Fu) << 4);
    return __builtin_bswap32(v);
#endif
}

IDB_HD int32_t idb_max(int32_t a, int32_t b) { return a > b ? a : b; }
IDB_HD int32_t idb_min(int32_t a, int32_t b) { return a < b ? a : b; }

// First mismatch at or after p (0 <= p <= b), at most b.
template <int W>
IDB_HD int32_t idb_slide(const uint32_t *m, int32_t p, int32_t b)
{
    const uint32_t cut = 0xFFFFFFFFu << ((uint32_t)p & 31u);
    uint32_t r = 0xFFFFFFFFu;
    if (W == 1) {
        r = idb_low_bit(m[0] & cut);  // (p = 32 = b: whatever it finds is raised to p)
    } else {
        const int32_t pw = p >> 5;
#pragma unroll
        for (int w = W - 1; w >= 0; --w) {
            const uint32_t v = w == pw ? m[w] & cut : m[w];
            const uint32_t at = idb_low_bit(v) | (uint32_t)(32 * w);
            r = w >= pw && at < r ? at : r;
        }
    }
    // clamp to [p, b]
    r = r > (uint32_t)b ? (uint32_t)b : r;
    return (int32_t)(r < (uint32_t)p ? (uint32_t)p : r);
}

// x and y: NP planes, plane p at word p * S, of which W words are looked at.
// Rows of at most 32 W letters, |lx - ly| <= t <= T (T >= 1); t < T only for T = 1, t = 0.
template <int NP, int W, int T, int S = W>
IDB_HD bool idb_lv_within(const uint32_t *x, const uint32_t *y, int32_t lx, int32_t ly, int32_t t)
{
    // y moved up T bits: diagonal d is then a right shift by d + T
    uint32_t ys[NP][W + 1];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        ys[p][0] = y[p * S] << T;
#pragma unroll
        for (int w = 1; w < W; ++w) ys[p][w] = idb_funnel(y[p * S + w], y[p * S + w - 1], 32 - T);
        ys[p][W] = y[p * S + W - 1] >> (32 - T);
    }
    const int32_t delta = ly - lx;
    // f of the level before, at index d + T; only |d| <= e are set
    int32_t f[2 * T + 1];
    uint32_t m[2 * T + 1][W];
    int32_t b[2 * T + 1];
#pragma unroll
    for (int d = -(T - 1); d <= T - 1; ++d) {
        const int k = d + T;
        b[k] = idb_min(lx, ly - d);
#pragma unroll
        for (int w = 0; w < W; ++w) {
            uint32_t v = x[w] ^ idb_funnel(ys[0][w + 1], ys[0][w], k);
#pragma unroll
            for (int p = 1; p < NP; ++p) v |= x[p * S + w] ^ idb_funnel(ys[p][w + 1], ys[p][w], k);
            m[k][w] = v;
        }
    }
    f[T] = idb_slide<W>(m[T], 0, idb_max(b[T], 0));
    if (T == 1 && t == 0) return delta == 0 && f[T] >= lx;
#pragma unroll
    for (int e = 1; e < T; ++e) {
        int32_t g[2 * T + 1];
#pragma unroll
        for (int d = -e; d <= e; ++d) {
            const int k = d + T;
            int32_t c = -1;
            if (d > -e && d < e) c = idb_max(c, f[k] + 1);       // substitution
            if (d - 1 > -e) c = idb_max(c, f[k - 1]);            // a letter of y
            if (d + 1 < e) c = idb_max(c, f[k + 1] + 1);         // a letter of x
            // (a diagonal that lies wholly outside has b < 0)
            const int32_t bb = idb_max(b[k], 0);
            g[k] = idb_slide<W>(m[k], idb_min(idb_max(c, 0), bb), bb);
        }
#pragma unroll
        for (int d = -e; d <= e; ++d) f[d + T] = g[d + T];
    }
    // the last level, on the diagonal the rows' ends lie on
    int32_t c = 0;
#pragma unroll
    for (int d = -T; d <= T; ++d) {
        const int k = d + T;
        int32_t v = 0;
        if (d > -T && d < T) v = f[k] + 1;
        if (d - 1 > -T) v = idb_max(v, f[k - 1]);
        if (d + 1 < T) v = idb_max(v, f[k + 1] + 1);
        c = delta == d ? v : c;
    }
    uint32_t md[W];
    const uint32_t s = (uint32_t)(delta + T) & 31u;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        uint32_t v = x[w] ^ idb_funnel(ys[0][w + 1], ys[0][w], s);
#pragma unroll
        for (int p = 1; p < NP; ++p) v |= x[p * S + w] ^ idb_funnel(ys[p][w + 1], ys[p][w], s);
        md[w] = v;
    }
    return idb_slide<W>(md, idb_min(c, lx), lx) >= lx;
}

// Rows of equal length: 1 = within t, 0 = not, 2 = idb_lv_within decides.  An
// alignment of equal rows has as many insertions as deletions, k each, and at
// most t - 2k substitutions.  k = 0 is the Hamming distance.  With t <= 3, k is
// at most 1: the rows are aligned on diagonal 0, then on +1 or -1 over x
// positions i1 .. i2, then on 0 again, with at most s = t - 2 substitutions.
// The first s + 1 mismatches of diagonal 0 reach into the middle, and so do
// the last s + 1; so the positions between them lie in it, and its diagonal
// mismatches there at most s times, once more for the position at its end
// that is not aligned.  Unrelated rows mismatch on three letters of four.
template <int NP, int W, int T, int S = W>
IDB_HD int idb_lv_equal_length(const uint32_t *x, const uint32_t *y, int32_t lx, int32_t t)
{
    uint32_t m[W], a[W], b[W];
    int h = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        uint32_t v = x[w] ^ y[w];
#pragma unroll
        for (int p = 1; p < NP; ++p) v |= x[p * S + w] ^ y[p * S + w];
        const int32_t in = idb_min(idb_max(lx - 32 * w, 0), 32);  // letters in this word
        m[w] = in == 32 ? v : v & ((1u << in) - 1u);
        h += __builtin_popcount(m[w]);
    }
    if (h <= t) return 1;
    if (T < 2) return 0;
    if (T > 3) return 2;
    // all bits from the (s + 1)-th lowest set bit up, and from the (s + 1)-th
    // highest down
#pragma unroll
    for (int dir = 0; dir < 2; ++dir) {
        uint32_t *r = dir ? b : a;
#pragma unroll
        for (int w = 0; w < W; ++w) r[w] = dir ? idb_reverse(m[W - 1 - w]) : m[w];
        if (T == 3) {  // clear the lowest set bit
            uint32_t bor = 1u;
#pragma unroll
            for (int w = 0; w < W; ++w) {
                const uint32_t v = r[w];
                r[w] = v & (v - bor);
                bor = v < bor ? 1u : 0u;
            }
        }
        uint32_t car = 1u;  // r | -r
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const uint32_t n = ~r[w] + car;
            car = car && n == 0u ? 1u : 0u;
            r[w] |= n;
        }
    }
    int up = 0, dn = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        const uint32_t in = a[w] & idb_reverse(b[W - 1 - w]);
        uint32_t u = 0, d = 0;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const uint32_t yw = y[p * S + w], hi = w + 1 < W ? y[p * S + w + 1] : 0u, lo = w > 0 ? y[p * S + w - 1] : 0u;
            u |= x[p * S + w] ^ idb_funnel(hi, yw, 1);
            d |= x[p * S + w] ^ idb_funnel(yw, lo, 31);
        }
        up += __builtin_popcount(u & in);
        dn += __builtin_popcount(d & in);
    }
    return up <= T - 1 || dn <= T - 1 ? 2 : 0;
}
