// idb_internal.h — device data layout and launch interfaces shared by the HIP
// translation units of libidb_hip.so.
//
// Layout in HBM for one run (all arrays device-resident, row = input row):
//   rows:     seq bytes, off[u64], len[u32], vbits[n*vw], jbits[n*jw]  (inputs)
//             key[u64]  duplicate hash, gslot[u32] the row's duplicate-table slot
//             rep[u32]  representative (min index of the duplicate class)
//             copies[u32], cnt[i32]  class size / exact neighbour count
//             par[u32]  union-find parent over rows, bmin[u32] border claim
//             pe[u32]   the entry that stands for the row, core flag in bit 31
//   duplicate table: P >= 2n slots of (smallest row, group size)
//   entries:  one per (unique row, V gene, J gene) bucket membership, sorted by
//             (repertoire, V gene, J gene, length, row); a bucket is a
//             contiguous run.  Per entry a 32-byte record (idb_entry, loaded
//             in one round trip) and the row's letters as dense 8-bit codes
//             (stride S bytes, S a multiple of 16) or, for Hamming mode,
//             packed words (stride HW words); for nucleotide rows a 3-gram
//             profile (64 saturating byte counts) per entry.
//   tiles:    (query block, target block) pairs of <= 64 entries each inside a
//             group (a bucket; in Hamming mode a bucket's run of one length)
//             whose length band can hold a neighbour pair.
//   edges:    neighbour pairs of the count pass in chunks of 2^chunk_log2
//             pairs; a wave fills one chunk at a time, chunk_fill[c] says how
//             many pairs chunk c holds.  Cluster growth rewrites them in place
//             as entry pairs.
//   entry forest: par_e[u32] union-find parent per entry, cmin_e[u32] the
//             smallest row of the component rooted at an entry.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "idb.h"

#define IDB_NONE 0xFFFFFFFFu
#define IDB_TILE 64               // entries per query / target block (one wave)
// Gene bitsets on the device: one header per gene name (its first 4 bytes
// and its last 4 bytes as little-endian words, zero-padded when shorter, its
// length, the offset of its 4-byte words in the packed name array).  A name
// that never matches (empty, or longer than 1024 bytes) has len = 0xFFFFFFFF.
struct idb_gene_hdr {
    uint32_t w0, w1, len, woff;
};
#define IDB_GENE_MAX_WIDTH 256u   // bit words per row (8,192 gene names)

// Entry order for runs of up to IDB_SORT_SMALL_MAX entries: stable radix
// sort of (u64 key, u32 value) pairs with the keys' low end_bit bits, two
// launches per digit pass (idb_sort.hip).  The sorted pairs end in (k1, v1)
// after an odd number of passes and back in (k0, v0) after an even one
// (*in_first); gcnt holds 256 counters per block.  hipErrorInvalidValue:
// sizes this sort does not take (nothing was launched).
#define IDB_SORT_SMALL_MAX (1u << 18)
// Single-launch exclusive scans and flag selection (idb_scan.hip).  The
// workspace (idb_scan_workspace_bytes for the largest n, zeroed when first
// allocated) holds a ticket counter and per-tile status words; launches on
// one workspace must be ordered (one stream), each with a generation the
// workspace has not seen since it was zeroed (1, 2, ...).  A look-back that
// did not end sets the 32-bit error word at idb_scan_error_offset().
size_t idb_scan_workspace_bytes(uint64_t max_n);
hipError_t idb_scan_exclusive_u32(const uint32_t *in, uint32_t *out, uint64_t n, void *ws, uint32_t gen, hipStream_t s);
hipError_t idb_scan_exclusive_u64(const uint64_t *in, uint64_t *out, uint64_t n, void *ws, uint32_t gen, hipStream_t s);
hipError_t idb_select_flagged(const uint8_t *flags, uint32_t *out, uint32_t *count, uint64_t n, void *ws, uint32_t gen,
                              hipStream_t s);
uint32_t idb_scan_error_offset();
uint32_t idb_sort_small_blocks(uint32_t n);
hipError_t idb_sort_small(uint64_t *k0, uint64_t *k1, uint32_t *v0, uint32_t *v1, uint32_t n, uint32_t end_bit,
                          uint32_t *gcnt, hipStream_t s, bool *in_first);

#define IDB_STAGE_BYTES 32768u    // each half of a context's pinned staging area
#define IDB_XFER_MAX_BYTES (256ull << 20)  // most pinned staging a context keeps for host inputs and outputs
// The run's small device words (zeroed at the start of a run): [12] chunks
// handed out, [16, 67) the depth histogram, [68, 88) time stamps, [100, 107)
// sizes for the host,
// then 8 copies of the row scan's 9 words (letter set, longest row) and 16
// partial counts each of core and noise rows (copies keep blocks from
// queueing their atomics on one word).
#define IDB_SMALL_ROWSCAN 128u
#define IDB_SMALL_CORES 200u
#define IDB_SMALL_NOISE 216u
#define IDB_SMALL_GENES 232u      // 8 copies of (highest V gene + 1, highest J gene + 1), row scan
#define IDB_SMALL_WORDS 256u
#define IDB_SMALL_READ (IDB_SMALL_GENES + 16u)  // words the host reads for the sizing
// The run's device counters: 8 64-bit statistics
#define IDB_WORK_U64 8u
// ... kept in IDB_WORK_COPIES copies (a kernel block adds into copy
// blockIdx & (copies - 1)), so that the waves' closing atomics do not queue
// on one word; readers sum the copies.
#define IDB_WORK_COPIES 16u
// Time stamps of the device's wall clock among the small words (a kernel's
// start or end: see idb_stamp_start); the counters behind the small words.
enum {
    IDB_T_BEGIN, IDB_T_DEDUP, IDB_T_UNIQ, IDB_T_TILES, IDB_T_COUNT, IDB_T_CORE, IDB_T_GROW, IDB_T_ROOTS, IDB_T_LABELS,
    IDB_T_END, IDB_N_STAMPS
};
#define IDB_SMALL_STAMPS 68u
#define IDB_SMALL_WORK IDB_SMALL_WORDS
#define IDB_SMALL_TOTAL (IDB_SMALL_WORK + 2u * IDB_WORK_U64 * IDB_WORK_COPIES)
// A run's results for the host in pinned memory (words): the small words, the
// counters' sums and the stamps, the scans' error word, the clusters, then the
// repertoires' first uniques.
#define IDB_FIN_WORK IDB_SMALL_WORDS
#define IDB_FIN_ERR (IDB_FIN_WORK + 64u)
#define IDB_FIN_CLUSTERS (IDB_FIN_ERR + 1u)
#define IDB_FIN_USTART (IDB_FIN_ERR + 16u)
#define IDB_FIN_USTART_MAX (IDB_STAGE_BYTES / 4u - IDB_FIN_USTART)
static_assert(2 * (IDB_WORK_U64 + IDB_N_STAMPS) <= 64 && IDB_SMALL_READ <= 256 && IDB_SMALL_STAMPS + 2 * IDB_N_STAMPS <= 100, "word layout");
#define IDB_MAX_W 8               // Myers 32-bit words per pattern (<= 256 letters)
#define IDB_MAX_HW 64             // Hamming packed words per row
#define IDB_MAX_LEN 65535u
#define IDB_ENC_P 32              // letters per row the encoder reads
#define IDB_QGRAM_WORDS 16        // 3-gram profile: 64 byte counts per row
#define IDB_QMASK_WORDS 8         // 3-gram level masks (learned runs): 3 x 64 bits, padded

struct idb_tile {
    uint32_t q0;                  // first query entry
    uint32_t t0;                  // first target entry
    uint32_t bucket;              // bucket id (gene pair) within its repertoire
    uint32_t shape;               // qn | tn << 8 | diag << 16
};

// Everything the pair kernels need about one entry, in one 32-byte record.
struct __align__(16) idb_entry {
    uint32_t row;                 // input row (a unique representative)
    uint32_t cp;                  // copies of the row
    uint32_t len_chk;             // length | chk << 16 (chk: the row may share a lower gene,
                                  // or every row in single-bucket mode)
    uint32_t t2;                  // threshold at this length: count pass (int16, low half),
                                  // fuse pass (int16, high half)
    uint32_t len;                 // the length alone (the second half is the count pass's
                                  // query record as it stands)
    uint32_t pres1, pres2;        // letters present at least once (the absent-letter filter) / twice
    uint32_t sig;                 // residues mod 16 of the genes the canonical test looks at:
                                  // V in the low half, J in the high half
};

// Uniform parameters of a pair-kernel launch.
struct idb_pair_args {
    const idb_tile *tiles;
    uint32_t n_tiles;
    const idb_entry *ent;
    const uint8_t *e_codes;       // Myers: stride S bytes of codes
    const uint32_t *e_pk;         // Hamming: stride HW packed words
    uint32_t S, HW, K;
    uint32_t bits;                // Hamming code width: 2, 5 or 8
    const int32_t *vbits, *jbits;
    uint32_t vw, jw;
    uint32_t gj;                  // J genes per bucket row (32*jw)
    uint32_t single_bucket;       // 1: every pair is gated explicitly
    uint32_t band_filter;         // 1: absent-letter filter before Myers (alphabets <= 31 letters)
    uint32_t qgram_filter;        // 1: 3-gram profile filter before Myers (alphabets <= 4 letters)
    const uint32_t *e_qg;         // 3-gram profiles, IDB_QGRAM_WORDS per entry
    const uint4 *e_low;           // per entry: its genes below the bucket's (V words, then J words), or null
    int32_t *cnt;                 // count pass output
    const int32_t *core;          // fuse pass input (per row)
    uint32_t *par;                // fuse pass: union-find parents
    uint32_t *bmin;               // fuse pass: border claims
    unsigned long long *work;     // [0] gated pairs, [1] neighbour pairs, [2] fuse pairs, [3] gated letters,
                                  // [5] Myers pairs, [6] Myers letters
    uint2 *edges;                 // count pass: neighbour pairs (x, y) in chunks, may be null
    uint32_t *chunk_fill;         // pairs written into each chunk
    uint32_t *n_chunks;           // chunks handed out (counts past max_chunks on overflow)
    uint32_t max_chunks;          // capacity in chunks
    uint32_t chunk_base;          // chunks 0 .. chunk_base - 1 belong to the waves of that number (counted in n_chunks)
    uint32_t chunk_log2;          // pairs per chunk = 1 << chunk_log2 (>= IDB_TILE)
    uint32_t fuse_if_overflow;    // fuse pass: run only when the pair list overflowed
    int32_t t_const;              // >= 0: every pair's count-pass threshold (absolute mode); -1 otherwise
    const uint16_t *zb;           // learned filter: bfloat16 embedding (64) per row
    float min_sim;                // learned filter: proposal threshold on z_x . z_y
    // matrix-core passes (idb_mx.hip), null otherwise: 4-bit features, length |
    // lower-gene flag << 16, records (protein rows: 5 planes, a spare word,
    // copies, length per entry; nucleotide rows: plane word w of entry e at
    // w * n_entries + e, then the copies), rows
    const uint32_t *e_feat, *e_meta, *e_vrec, *e_row;
    uint32_t n_entries;
    uint32_t mx_planes, mx_words; // planes per letter (5 or 2), words per plane
    int32_t *cnt_e;               // their count output, per entry; their pair list holds entries
    uint32_t sub_log2;            // tiles are taken in 2^sub_log2 parts of their queries
    // launch shape (0 = default): waves per block, grid = resident blocks x
    // grid_mul, and plain block order instead of the XCD-grouped one
    uint32_t tune_wpb, tune_grid_mul, no_xcd_order;
};

// Time stamps inside kernels: at the start by the first block, at the end by
// one block in 32 (the latest counts).
__device__ __forceinline__ void idb_stamp_start(unsigned long long *at)
{
    if (at && blockIdx.x == 0 && threadIdx.x == 0) *at = wall_clock64();
}
__device__ __forceinline__ void idb_stamp_end(unsigned long long *at)
{
    if ((blockIdx.x & 31u) == 0 && threadIdx.x == 0) atomicMax(at, (unsigned long long)wall_clock64());
}

// Bytes k .. k+15 of a row of length L as one 16-byte value, zero past the
// row's end (k a multiple of 16).  Every load stays inside the row: a short
// tail is read as the row's last 16 bytes and shifted down, a row of 8 to 15
// bytes as its first and its last eight, shorter rows byte by byte.  Unaligned
// global loads are legal on gfx950.
// Only 32-bit shifts: a 64-bit shift whose amount the compiler puts into the
// last of a wave's vector registers now and then comes out wrong, and one
// kernel was compiled so (the gene scan with a 32-bit table and bit words in
// memory: of 400,000 rows, 600 to 750 lost the name at their end).
// tests/test_code_objects.py looks for it.  Against 64-bit shifts and bytes for
// all rows under 16 (the kernels that read rows this way, us): 2.56M nucleotide
// rows 690 -> 680, 2M protein rows 535 -> 427, 2M long nucleotide rows 794 -> 789,
// 1M gene calls 51.7 -> 50.9.
__device__ __forceinline__ uint4 row16(const uint8_t *s, uint32_t L, uint32_t k)
{
    uint4 v;
    if (k + 16 <= L) {
        __builtin_memcpy(&v, s + k, 16);
        return v;
    }
    if (L >= 16) {
        __builtin_memcpy(&v, s + L - 16, 16);
        const uint32_t d = 16 - (L - k);  // bytes to drop
        if (d & 8u) v = make_uint4(v.z, v.w, 0u, 0u);
        if (d & 4u) v = make_uint4(v.y, v.z, v.w, 0u);
        return make_uint4(__builtin_amdgcn_alignbyte(v.y, v.x, d), __builtin_amdgcn_alignbyte(v.z, v.y, d),
                          __builtin_amdgcn_alignbyte(v.w, v.z, d), __builtin_amdgcn_alignbyte(0u, v.w, d));
    }
    if (L >= 8) {
        uint32_t h[2], t[2];
        __builtin_memcpy(h, s, 8);
        __builtin_memcpy(t, s + L - 8, 8);
        const uint32_t d = 16 - L, x = d & 4u ? t[1] : t[0], y = d & 4u ? 0u : t[1];
        return make_uint4(h[0], h[1], L > 8 ? __builtin_amdgcn_alignbyte(y, x, d) : 0u,
                          L > 8 ? __builtin_amdgcn_alignbyte(0u, y, d) : 0u);
    }
    v = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll 1
    for (uint32_t b = 0; b < L; ++b) {
        const uint32_t c = (uint32_t)s[b] << (8 * (b & 3u));
        v.x |= b < 4 ? c : 0u;
        v.y |= b < 4 ? 0u : c;
    }
    return v;
}

__device__ __forceinline__ uint32_t byte_of(const uint4 &v, uint32_t b)
{
    const uint32_t w = b < 8 ? (b < 4 ? v.x : v.y) : (b < 12 ? v.z : v.w);
    return (w >> (8 * (b & 3))) & 0xFFu;
}

// Word k of a gene bitset restricted to the genes below gene g.
__device__ __forceinline__ uint32_t below_gene(uint32_t w, uint32_t k, uint32_t g)
{
    if (k * 32 >= g) return 0u;
    return (k * 32 + 32 > g) ? (w & ((1u << (g - k * 32)) - 1u)) : w;
}

// Counts one more 3-gram (0..63) in the level masks of a nucleotide row:
// g[2k], g[2k+1] = the 3-grams seen at least k + 1 times, k = 0, 1, 2.
__device__ __forceinline__ void idb_qmask_add(uint32_t (&g)[6], uint32_t gram)
{
    const uint32_t bit = 1u << (gram & 31u), lo = gram < 32u ? bit : 0u, hi = gram < 32u ? 0u : bit;
    g[4] |= g[2] & lo;
    g[5] |= g[3] & hi;
    g[2] |= g[0] & lo;
    g[3] |= g[1] & hi;
    g[0] |= lo;
    g[1] |= hi;
}

// LDS bytes one wave of the Myers kernels needs: Peq columns, the edge
// staging slots, the Myers queue (2 * IDB_TILE 16-bit entries), the per-tile
// count accumulators of queries and targets, and the tile's query records.
__host__ __device__ inline size_t idb_myers_lds_per_wave(uint32_t K, uint32_t W)
{
    return ((size_t)K * W * 64 + 2 * IDB_TILE + IDB_TILE + 2 * IDB_TILE) * sizeof(uint32_t) +
           IDB_TILE * sizeof(idb_entry);
}
// Extra LDS per wave for the query profiles of the 3-gram filter.
__host__ __device__ inline size_t idb_qgram_lds_per_wave() { return (size_t)IDB_TILE * IDB_QGRAM_WORDS * sizeof(uint32_t); }
// The device's LDS limit per block (opt-in value where the device has one).
size_t idb_lds_limit();

// Kernel launchers (defined in idb_pairs.hip).
hipError_t idb_launch_count_myers(const idb_pair_args &a, uint32_t W, hipStream_t s);
hipError_t idb_launch_fuse_myers(const idb_pair_args &a, uint32_t W, hipStream_t s);
hipError_t idb_launch_count_hamming(const idb_pair_args &a, hipStream_t s);
hipError_t idb_launch_fuse_hamming(const idb_pair_args &a, hipStream_t s);
hipError_t idb_launch_count_learned(const idb_pair_args &a, hipStream_t s);
hipError_t idb_launch_pair_distances(const uint8_t *seq, const uint64_t *off, const uint32_t *len, const uint2 *pairs,
                                     unsigned long long n, uint32_t W, uint32_t ham, uint32_t *dist, hipStream_t s);
// The matrix-core count and fuse passes (idb_mx.hip) and their entry arrays.
#define IDB_MX_MAX_LETTERS 30u    // alphabet of the one-word (protein) form
struct idb_mx_fill_args {
    const uint64_t *ekey;
    const uint32_t *erow;
    uint32_t E;
    const uint8_t *seq;
    uint32_t vw, jw, gj, gvj;
    const uint8_t *cmap;
    uint32_t planes, K, W;
    int32_t t;
    uint32_t lb;
    uint16_t *elen;
    uint32_t *meta, *feat, *vrec;
    uint8_t *bflag;
    uint32_t *inv;                // entry of each (row, gene pair), rows in order (first index: row record word 3)
    int32_t *cnt_e;
    uint32_t *par_e, *cmin_e;
    uint4 *elow;
    const uint4 *rrec;
};
struct idb_mx_rows_args {
    const uint32_t *uniq, *num;
    const uint64_t *eoff;
    const uint32_t *inv;
    const int32_t *cnt_e;
    const uint32_t *copies;
    uint32_t n;
    int32_t min_pts;
    int32_t *cnt, *core;
    uint32_t *pe;
    uint8_t *ecore;
    uint32_t *par_e, *n_cores;
    unsigned long long *stamps;
};
hipError_t idb_launch_mx_fill(const idb_mx_fill_args &f, hipStream_t s);
hipError_t idb_launch_mx_rows(const idb_mx_rows_args &r, hipStream_t s);
hipError_t idb_launch_mx_count(const idb_pair_args &a, hipStream_t s);
hipError_t idb_launch_mx_fuse(const idb_pair_args &a, hipStream_t s);
// Launch helpers (idb_pairs.hip).
uint32_t idb_resident_blocks(const void *kernel, uint32_t block, size_t shm);
uint32_t idb_grid_for(uint32_t n_tiles, uint32_t wpb, uint32_t resident, uint32_t mul);
uint32_t idb_count_grid(const idb_pair_args &a, uint32_t n_tiles, uint32_t wpb, uint32_t resident);
uint32_t idb_pick_wpb(const idb_pair_args &a, uint32_t most);
hipError_t idb_launch_gene_bitsets(const uint8_t *calls, const uint64_t *off, const uint32_t *len, uint32_t n,
                                   const idb_gene_hdr *hdr, const uint32_t *gw, uint32_t n_words, uint32_t n_genes,
                                   int32_t *out, uint32_t width, hipStream_t s);
hipError_t idb_launch_gene_scan(const uint8_t *calls, const uint64_t *off, const uint32_t *len, uint32_t n,
                                const uint8_t *cls, const uint32_t *nodes, const void *trans, bool narrow,
                                uint32_t ncls, uint32_t entries, uint32_t out_min, uint32_t n_nodes, uint32_t max_len,
                                int32_t *out, uint32_t width, hipStream_t s);
// Cluster growth over the count pass's pairs (rewrites the pair list in place).
struct idb_union_args {
    const uint32_t *pe;           // per row: one of its entries | core flag << 31; IDB_NONE without entries
    uint32_t *par_e;              // per entry: union-find parent, its own index on entry
    uint32_t *cmin_e;             // per entry: smallest row of the component rooted there, IDB_NONE on entry
    uint32_t n_entries, n_rows;
    uint32_t *par;                // per row: set to the component minimum for core rows
    uint32_t *bmin;               // per row: border claims
    const uint32_t *rep;          // per row: representative (for the depth histogram)
    const uint8_t *ecore;         // per entry: its row's core flag, when the pair list holds entries (else null)
    const uint32_t *erow;         // per entry: its row
    uint32_t *depth_hist;         // 51 bins of union-find depths, or null (no histogram)
};
hipError_t idb_launch_union_edges(const idb_pair_args &a, const idb_union_args &u, hipStream_t s);

// Encoder (idb_learned.hip): bfloat16 embeddings of rows [0, n) on stream s.
struct idb_encoder;
hipError_t idb_encoder_embed_rows(idb_encoder *e, const uint8_t *seq, const uint64_t *off, const uint32_t *len,
                                  uint32_t n, uint16_t *zb, hipStream_t s);
const char *idb_encoder_error(const idb_encoder *e);
int idb_encoder_device(const idb_encoder *e);
