// gene_table.h — the multi-name automaton of the gene-call scan (host code).
//
// A. V. Aho and M. J. Corasick ("Efficient string matching: an aid to
// bibliographic search", CACM 1975) over the gene names: one pass over a call
// string's bytes, one table lookup per byte, finds every name that occurs in
// it.  Bytes are first mapped to classes (class 0: bytes that occur in no
// name, which lead back to the root), so that a row of the table holds one
// entry per class instead of 256.
//
// A table row is the state's `ncls` transitions and then its list head
// (stride = ncls + 1).  A transition is the target row's offset in entries
// (state * stride).  States at which some name ends are numbered last: their
// offsets are out_min and above, so that the walk needs no flag bits.  The
// list head is 0 or 1 + the index of the first node of the names that end at
// the state: node = gene | next << 16, next in the same encoding; a state's
// own names come first and are followed by its suffix states'.
//
// Byte 0 is always in class 0, so that a walk may run over zero bytes past a
// string's end: names that hold a zero byte are not taken.
#pragma once
#include <stdint.h>

#include <algorithm>
#include <cstddef>
#include <vector>

struct idb_gene_table {
    uint32_t ncls = 0, stride = 0, entries = 0;
    uint32_t out_min = 0;           // offset of the first state that ends a name (entries: none)
    uint32_t max_len = 0;           // longest usable name
    uint8_t cls[256] = {};          // class of a byte value
    std::vector<uint32_t> trans;
    std::vector<uint32_t> nodes;
};

#define IDB_GENE_NAME_MAX 1024u         // longer names never match
#define IDB_GENE_TABLE_NARROW 32768u    // entries of a table that goes to LDS (16-bit byte offsets)
#define IDB_GENE_TABLE_MAX (1u << 20)   // entries of the largest table that is built

// The automaton while building its table costs less than testing every name:
// measured, the per-name kernel takes 0.45 us per name (a wave's walk over the
// names) + 0.081 ns per call and name, the automaton about 11 us + 4.5 ns per
// table entry (mostly its construction on the host).  104 V genes: 58 against
// 70 us from 100 calls on, 74 us against 8.75 ms at 1M; 37 D genes: even at
// 5,000 calls; 6 J genes: from about 15,000 calls (31.5 against 36.6 us at
// 20,000).  The largest table that is worth building for n calls:
inline uint32_t idb_gene_table_cap(uint32_t n, uint32_t n_genes)
{
    const int64_t worth = 100ll * n_genes + (int64_t)((uint64_t)n * n_genes * 18u / 1000u) - 2500;
    return (uint32_t)std::max<int64_t>(0, std::min<int64_t>(IDB_GENE_TABLE_MAX, worth));
}

// Letters of name b past its common prefix with name a (of which 64 letters are
// looked at).
inline uint32_t idb_gene_fresh(const uint8_t *a, uint32_t la, const uint8_t *b, uint32_t lb)
{
    const uint32_t most = std::min(std::min(la, lb), 64u);
    uint32_t k = 0;
    while (k < most && a[k] == b[k]) ++k;
    return lb - k;
}

// False when a table of at most cap entries is out of reach, by a look at up to
// 64 names: a build that is given up at the cap costs most of a finished one
// (8,000 random names of 8 to 12 letters 0.4 ms of a 1.07 ms call, 64 of about
// 1,000 letters 25 us of 53).  States per name are taken from the letters that a
// name adds to the one before it in the list (lists in order), and, when those
// are too many, to the one before it among the sorted sample.  Both count too
// many states where more names share prefixes than the look shows, hence the
// factor (measured too many by 1.0 to 1.5: gene lists in order and shuffled,
// random names).
inline bool idb_gene_table_in_reach(uint32_t n_genes, const uint8_t *genes, const uint64_t *gene_off,
                                    const uint32_t *gene_len, uint32_t cap)
{
    uint32_t at[64], n = 0, classes = 0;
    bool seen[256] = {};
    uint64_t fresh = 0, pairs = 0;
    const auto usable = [&](uint32_t g) { return gene_len[g] != 0 && gene_len[g] <= IDB_GENE_NAME_MAX; };
    const auto added = [&](uint32_t a, uint32_t b) {
        return idb_gene_fresh(genes + gene_off[a], gene_len[a], genes + gene_off[b], gene_len[b]);
    };
    const auto reach = [&](double per_name) { return per_name * n_genes * (classes + 2u) <= 1.3 * cap; };
    uint64_t letters = 1;  // a state per letter and an entry per byte value are the most there can be
    for (uint32_t g = 0; g < n_genes; ++g) letters += usable(g) ? gene_len[g] : 0u;
    if (letters * 257u <= cap) return true;
    const uint32_t step = (n_genes + 63u) / 64u;
    for (uint32_t g = step / 2; g < n_genes; g += step) {
        if (!usable(g)) continue;
        at[n++] = g;
        for (uint32_t k = 0; k < gene_len[g] && k < 16u; ++k) {
            classes += !seen[genes[gene_off[g] + k]];
            seen[genes[gene_off[g] + k]] = true;
        }
        if (g && usable(g - 1u)) {
            fresh += added(g - 1u, g);
            ++pairs;
        }
    }
    if (n < 2 || pairs == 0 || reach((double)fresh / pairs)) return true;
    std::sort(at, at + n, [&](uint32_t a, uint32_t b) {
        return std::lexicographical_compare(genes + gene_off[a], genes + gene_off[a] + gene_len[a],
                                            genes + gene_off[b], genes + gene_off[b] + gene_len[b]);
    });
    fresh = 0;
    for (uint32_t k = 1; k < n; ++k) fresh += added(at[k - 1], at[k]);
    return reach((double)fresh / (n - 1));
}

// LDS of a block that keeps the table there: class map, 16-bit entries, nodes.
inline size_t idb_gene_table_lds(const idb_gene_table &t)
{
    return 256 + ((size_t)t.entries + 1) / 2 * 4 + 4 * t.nodes.size();
}

// True for a table that goes to LDS (of which a block may have lds_limit bytes).
inline bool idb_gene_table_narrow(const idb_gene_table &t, size_t lds_limit)
{
    return t.entries <= IDB_GENE_TABLE_NARROW && t.nodes.size() <= 4096 && idb_gene_table_lds(t) <= lds_limit;
}

// False when the table would hold more than `cap` entries or a name holds a
// zero byte.
inline bool idb_gene_table_build(uint32_t n_genes, const uint8_t *genes, const uint64_t *gene_off,
                                 const uint32_t *gene_len, uint32_t cap, idb_gene_table &t)
{
    t = idb_gene_table();
    t.ncls = 1;
    for (uint32_t g = 0; g < n_genes; ++g) {
        const uint32_t L = gene_len[g];
        if (L == 0 || L > IDB_GENE_NAME_MAX) continue;
        if (L > t.max_len) t.max_len = L;
        for (uint32_t k = 0; k < L; ++k) {
            const uint8_t b = genes[gene_off[g] + k];
            if (!b) return false;
            if (!t.cls[b]) t.cls[b] = (uint8_t)t.ncls++;  // (at most 255 values)
        }
    }
    const uint32_t st = t.stride = t.ncls + 1u;
    if (st > cap) return false;
    t.trans.reserve(std::min<size_t>(cap, 8192u));
    t.trans.assign(st, 0u);
    std::vector<uint32_t> tail;  // per state: 1 + its own last node, 0 without
    tail.push_back(0u);
    uint32_t states = 1;
    for (uint32_t g = 0; g < n_genes; ++g) {
        const uint32_t L = gene_len[g];
        if (L == 0 || L > IDB_GENE_NAME_MAX) continue;
        uint32_t s = 0;
        for (uint32_t k = 0; k < L; ++k) {
            const size_t at = (size_t)s * st + t.cls[genes[gene_off[g] + k]];
            if (!t.trans[at]) {
                if ((uint64_t)(states + 1u) * st > cap) return false;
                t.trans[at] = states++;
                t.trans.resize((size_t)states * st, 0u);
                tail.push_back(0u);
            }
            s = t.trans[at];
        }
        t.nodes.push_back(g);
        uint32_t &head = t.trans[(size_t)s * st + t.ncls];
        if (tail[s]) t.nodes[tail[s] - 1u] |= (uint32_t)t.nodes.size() << 16;
        else head = (uint32_t)t.nodes.size();
        tail[s] = (uint32_t)t.nodes.size();
    }
    t.entries = states * st;
    // breadth first: missing edges from the suffix state's finished row, and
    // the suffix state's list behind the state's own
    std::vector<uint32_t> fail(states, 0u), queue;
    queue.reserve(states);
    for (uint32_t c = 0; c < t.ncls; ++c)
        if (t.trans[c]) queue.push_back(t.trans[c]);
    for (size_t q = 0; q < queue.size(); ++q) {
        const uint32_t s = queue[q];
        uint32_t *row = &t.trans[(size_t)s * st];
        const uint32_t *frow = &t.trans[(size_t)fail[s] * st];
        for (uint32_t c = 0; c < t.ncls; ++c) {
            if (row[c]) {
                fail[row[c]] = frow[c];
                queue.push_back(row[c]);
            } else {
                row[c] = frow[c];
            }
        }
        if (tail[s]) t.nodes[tail[s] - 1u] |= frow[t.ncls] << 16;
        else row[t.ncls] = frow[t.ncls];
    }
    // states without a name to report first, then the others
    std::vector<uint32_t> at(states);
    uint32_t quiet = 0, loud = 0;
    for (uint32_t s = 0; s < states; ++s) quiet += t.trans[(size_t)s * st + t.ncls] == 0u;
    t.out_min = quiet * st;
    loud = quiet;
    quiet = 0;
    for (uint32_t s = 0; s < states; ++s) at[s] = (t.trans[(size_t)s * st + t.ncls] ? loud++ : quiet++) * st;
    std::vector<uint32_t> out(t.entries);
    for (uint32_t s = 0; s < states; ++s) {
        const uint32_t *from = &t.trans[(size_t)s * st];
        uint32_t *to = &out[at[s]];
        for (uint32_t c = 0; c < t.ncls; ++c) to[c] = at[from[c]];
        to[t.ncls] = from[t.ncls];
    }
    t.trans.swap(out);
    return true;
}
