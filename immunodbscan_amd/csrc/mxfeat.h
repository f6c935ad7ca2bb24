// mxfeat.h — the 4-bit feature vectors of the matrix-core count pass
// (idb_mx.hip), shared with a host-side test.
//
// A row's features are bits: "letter c occurs at least k times" (protein rows,
// k = 1, 2) or "3-gram g occurs at least k times" (nucleotide rows, k = 1, 2,
// 3).  One edit removes at most one letter occurrence and adds at most one
// (at most three 3-grams each: E. Ukkonen, "Approximate string-matching with
// q-grams and maximal matches", TCS 1992), so with nx = |x|, ny = |y| set
// features and dot = |x and y|,
//   lev(x, y) <= t   implies   nx - dot <= s t  and  ny - dot <= s t
// (s = 1 for letters, 3 for 3-grams; leaving features out keeps it true).
// As 4-bit floats (E2M1) the dot product is exact on the matrix cores.  The
// last dimensions carry the row's own term s t - n as digits against fixed
// weights (6 and 1) on the other side, so that one product gives
// dot + s t - nx and another dot + s t - ny: a pair passes when neither is
// negative.
#pragma once
#include <stdint.h>

#ifndef IDB_HD
#if defined(__HIPCC__)
#define IDB_HD __host__ __device__ __forceinline__
#else
#define IDB_HD static inline
#endif
#endif

// Protein rows: 64 dimensions, 60 letter bits (two per letter, at most 30
// letters), two digits of weight 6 and two of weight 1: |s t - n| <= 35 fits,
// n <= 32 (rows of at most 32 letters), t <= 3.
// Nucleotide rows: 192 dimensions, 64 + 64 + 56 3-gram bits (the last eight
// 3-grams have no third bit), six digits of weight 6 and two of weight 1:
// |s t - n| <= 185 fits (30 sixes and 5), n <= 184, t <= 4.
#define IDB_MX_AA_WEIGHTS 0x2277u       // dims 60..63
#define IDB_MX_NT_WEIGHTS 0x22777777u   // dims 184..191
#define IDB_MX_NT_L3HI 0x00FFFFFFu      // third-level bits of 3-grams 32..63 that exist

// Bits 0..7 as eight 4-bit ones (E2M1 1.0 = 0b0010).
IDB_HD uint32_t idb_mx_spread(uint32_t b)
{
    uint32_t x = b & 0xFFu;
    x = (x | (x << 12)) & 0x000F000Fu;
    x = (x | (x << 6)) & 0x03030303u;
    x = (x | (x << 3)) & 0x11111111u;
    return x << 1;
}

// n digits in {0, 1, 2, 3, 4, 6} that sum to v, as E2M1 codes (lowest first).
IDB_HD uint32_t idb_mx_sum(uint32_t v, uint32_t n, uint32_t sign)
{
    uint32_t out = 0;
    for (uint32_t k = 0; k < n; ++k) {
        const uint32_t d = v >= 6 ? 6u : (v >= 4 ? 4u : v);
        const uint32_t code = d == 6 ? 7u : (d == 4 ? 6u : (d == 3 ? 5u : 2u * d));
        out |= (d ? code | sign : 0u) << (4 * k);
        v -= d;
    }
    return out;
}

// v = 6 a + b as n6 digits of weight 6 and two of weight 1.
IDB_HD uint32_t idb_mx_digits(int32_t v, uint32_t n6)
{
    const uint32_t sign = v < 0 ? 8u : 0u, m = (uint32_t)(v < 0 ? -v : v);
    return idb_mx_sum(m / 6u, n6, sign) | (idb_mx_sum(m % 6u, 2, sign) << (4 * n6));
}
