// R2 gene bitsets on the device: bit g of row i is set iff gene name g occurs
// as a contiguous substring of call string i (cuda/BitsetVector.inl:151-175).
// The reference launches one grid per gene (find_string_occurences,
// cuda/BitsetVector.inl:181-209).  Two kernels here:
//
// k_gene_scan walks the multi-name automaton of gene_table.h, one call string
// per lane, one table lookup per byte whatever the number of names.  The
// table sits in LDS as 16-bit entries when it has at most 32,768 (104 V gene
// names make 7,248 entries, 14.5 KB), else in global memory as 32-bit
// ones.
//
// k_gene_bitsets, where building the table would cost more than it saves (few
// names and calls, or very long names): one wave takes one call string
// and tests every gene against it:
//   * the string is staged in the wave's LDS window, 2048 bytes at a time,
//     with start positions advancing 1024 at a time (names longer than 1024
//     bytes never match, as in the reference whose launch of more than 1024
//     threads fails), so every start position sees its whole candidate;
//   * lane p holds the 4 bytes at start position p (v_alignbyte of two LDS
//     words); a name's first 4 bytes are compared with one masked XOR and
//     its last 4 bytes with one more (gene names share their first bytes:
//     every IGHV name starts "IGHV"), and the lanes that pass check the
//     middle of the name 4 bytes at a time;
//   * the gene headers (the first 512) and the name words (when they fit in
//     2048 words) are staged in LDS once per block and read by broadcast; the
//     row's bit words collect in LDS and leave with one store per word.
#include <algorithm>

#include "idb_internal.h"
#include "gene_table.h"

namespace {

constexpr uint32_t GS_LONG = 2048;           // longer call strings may be walked by a whole wave
constexpr uint32_t GS_LANE = 1u << 20;       // ... and still longer ones always are

// A lane's walk over one call string, with offsets in bytes (one add-shift
// per lookup).  A byte where a name ends only notes the state, in a queue of
// four in registers pushed without a branch; the queue is emptied when a
// lane's is full and at the end of the string.  (Following the lists at once
// costs the whole wave their latency at nearly every byte: with two alleles
// per call some lane has one.)  NW > 0: the row's bit words are in w[];
// NW == 0: they are in global memory (atomic, so that several lanes may walk
// one row).
template <typename TE, int NW>
struct GeneWalk {
    static constexpr int SH = sizeof(TE) == 2 ? 1 : 2;
    const char *tr;
    const uint8_t *cls;
    const uint32_t *nodes;
    uint32_t head_at, out_min;    // byte offsets: list head within a row, first state that ends a name
    int32_t *out;                 // NW == 0: the row's words
    uint32_t s = 0, cnt = 0;
    uint32_t q[4] = {};           // the states noted, newest first (16-bit tables: two per word)
    uint32_t w[NW ? NW : 1] = {};

    __device__ __forceinline__ uint32_t at(uint32_t o) const { return *(const TE *)(tr + o); }
    __device__ __forceinline__ void flush()
    {
        for (; cnt; --cnt) {
            uint32_t st;
            if (sizeof(TE) == 2) {
                st = q[0] & 0xFFFFu;
                q[0] = __builtin_amdgcn_alignbit(q[1], q[0], 16);
                q[1] >>= 16;
            } else {
                st = q[0];
                q[0] = q[1];
                q[1] = q[2];
                q[2] = q[3];
            }
            for (uint32_t n = at(st + head_at); n;) {
                const uint32_t v = nodes[n - 1u], g = v & 0xFFFFu, bit = 1u << (g & 31u);
                n = v >> 16;
                if (NW) {
#pragma unroll
                    for (int k = 0; k < NW; ++k)
                        if ((g >> 5) == (uint32_t)k) w[k] |= bit;
                } else {
                    atomicOr((uint32_t *)out + (g >> 5), bit);
                }
            }
        }
    }
    __device__ __forceinline__ void step(uint32_t byte)
    {
        s = at(s + ((uint32_t)cls[byte] << SH));
        if (cnt == 4u) flush();
        const bool end = s >= out_min;
        if (sizeof(TE) == 2) {
            const uint32_t hi = __builtin_amdgcn_alignbit(q[1], q[0], 16), lo = (q[0] << 16) | s;
            q[1] = end ? hi : q[1];
            q[0] = end ? lo : q[0];
        } else {
#pragma unroll
            for (int k = 3; k > 0; --k) q[k] = end ? q[k - 1] : q[k];
            q[0] = end ? s : q[0];
        }
        cnt += end ? 1u : 0u;
    }
};

// One call string per lane.  The bound is the chain of dependent lookups (a
// byte's row depends on the byte before), so the chip is filled with as many
// lanes as fit; neighbouring lanes read neighbouring strings 16 bytes at a
// time, so every line of the calls is fetched once.  1M calls of 46.7 bytes
// against 104 names: 8,666 us for the per-name kernel, 51 us here (20M VALU
// wave instructions, 33 us of issue; 47 MB of calls at the copy rate: 14 us).
// A string longer than GS_LONG is cut into 64 segments walked by the lanes of
// its wave, each starting max_len - 1 bytes early at the root state (a name
// that ends in the segment starts no earlier), where that is the shorter way:
// the wave walks its long strings one after the other, at twice the time per
// byte (it reads byte by byte), while a string per lane runs beside the
// others'.  104 V genes, strings of 2,100 bytes: a single one 39 us a call by
// the wave, 100 of them 541 us that way and 179 a lane each; 1,000 of 40,000
// bytes 12.4 and 3.0 ms.
template <typename TE, int NW>
__global__ __launch_bounds__(1024) void k_gene_scan(const uint8_t *calls, const uint64_t *off, const uint32_t *len,
                                                    uint32_t n, const uint8_t *__restrict__ cls_g,
                                                    const TE *__restrict__ tr_g, const uint32_t *__restrict__ nodes_g,
                                                    uint32_t ncls, uint32_t entries, uint32_t out_min, uint32_t n_nodes,
                                                    uint32_t max_len, int32_t *out, uint32_t width,
                                                    uint32_t wide_store)
{
    extern __shared__ uint32_t gs_lds[];
    constexpr bool IN_LDS = sizeof(TE) == 2;
    const uint8_t *cls = (const uint8_t *)gs_lds;        // 256 bytes, then the table
    for (uint32_t k = threadIdx.x; k < 64; k += blockDim.x) gs_lds[k] = ((const uint32_t *)cls_g)[k];
    if (IN_LDS)
        for (uint32_t k = threadIdx.x; k < (entries + 1) / 2; k += blockDim.x)
            gs_lds[64 + k] = ((const uint32_t *)tr_g)[k];
    // (16-bit tables: the nodes follow in LDS)
    uint32_t *nodes_l = gs_lds + 64 + (entries + 1) / 2;
    if (IN_LDS)
        for (uint32_t k = threadIdx.x; k < n_nodes; k += blockDim.x) nodes_l[k] = nodes_g[k];
    __syncthreads();
    const char *tr = IN_LDS ? (const char *)(gs_lds + 64) : (const char *)tr_g;
    const uint32_t head_at = ncls * sizeof(TE), out_b = out_min * sizeof(TE);
    const uint32_t *nodes = IN_LDS ? nodes_l : nodes_g;
    const uint32_t lane = __lane_id();
    const uint32_t step = gridDim.x * blockDim.x;
    // whole waves stay together: `base` is the wave's first row
    for (uint32_t base = blockIdx.x * blockDim.x + (threadIdx.x & ~63u); base < n; base += step) {
        const uint32_t row = base + lane;
        const bool valid = row < n;
        const uint32_t L = valid ? len[row] : 0u;
        const uint8_t *src = calls + (valid ? off[row] : 0ull);
        int32_t *ro = out + (size_t)row * width;
        if (!NW && valid)
            for (uint32_t k = 0; k < width; ++k) ro[k] = 0;
        bool is_long = L > GS_LONG;
        if (const uint64_t lm = __ballot(is_long)) {
            uint32_t longest = L;
#pragma unroll
            for (int d = 32; d > 0; d >>= 1) longest = max(longest, (uint32_t)__shfl_xor((int)longest, d, 64));
            const uint64_t by_wave = 2ull * (uint32_t)__popcll(lm) * (longest / 64u + max_len);
            is_long = is_long && (longest > GS_LANE || by_wave < longest);
        }
        if (!NW) __threadfence();  // the zeros are in place before any bit is set
        GeneWalk<TE, NW> wk{tr, cls, nodes, head_at, out_b, ro};
        if (!is_long) {
            uint4 nx = L ? row16(src, L, 0) : make_uint4(0, 0, 0, 0);
            for (uint32_t k0 = 0; k0 < L; k0 += 16) {
                const uint4 v = nx;
                if (k0 + 16 < L) nx = row16(src, L, k0 + 16);
                // bytes past the string's end are zero and lead to the root
#pragma unroll
                for (uint32_t b = 0; b < 16; ++b) wk.step(byte_of(v, b));
            }
            wk.flush();
        }
        for (uint64_t lm = __ballot(is_long); lm; lm &= lm - 1ull) {
            const int o = __builtin_ctzll(lm);
            const uint32_t Lo = (uint32_t)__shfl((int)L, o, 64);
            const uint64_t so = __shfl((unsigned long long)(valid ? off[row] : 0ull), o, 64);
            const uint32_t seg = (Lo + 63u) / 64u;
            const uint64_t a = (uint64_t)lane * seg, e = min((uint64_t)Lo, a + seg);
            GeneWalk<TE, NW> lw{tr, cls, nodes, head_at, out_b, out + (size_t)(base + (uint32_t)o) * width};
            for (uint64_t k = a > max_len - 1u ? a - (max_len - 1u) : 0u; k < e; ++k) lw.step(calls[so + k]);
            lw.flush();
            if (NW) {
#pragma unroll
                for (int k = 0; k < NW; ++k) {
#pragma unroll
                    for (int d = 32; d > 0; d >>= 1) lw.w[k] |= (uint32_t)__shfl_xor((int)lw.w[k], d, 64);
                    if ((int)lane == o) wk.w[k] = lw.w[k];
                }
            }
        }
        const uint32_t *w = wk.w;
        if (NW && valid) {
            if (NW == 4 && wide_store) {
                *(uint4 *)ro = make_uint4(w[0], w[1], w[2], w[3]);
            } else {
#pragma unroll
                for (int k = 0; k < NW; ++k)
                    if ((uint32_t)k < width) ro[k] = (int32_t)w[k];
            }
        }
    }
}

constexpr uint32_t GSEG = 1024;              // start positions per window
constexpr uint32_t GWIN = 2 * GSEG;          // window bytes
constexpr uint32_t GWIN_WORDS = GWIN / 4 + 4;
constexpr uint32_t GWPB = 4;                 // waves per block
constexpr uint32_t GHDR_LDS = 512;           // gene headers kept in LDS
constexpr uint32_t GW_LDS = 2048;            // name words kept in LDS

__device__ __forceinline__ uint32_t win_word(const uint32_t *win, uint32_t b)
{
    return __builtin_amdgcn_alignbyte(win[(b >> 2) + 1], win[b >> 2], b & 3u);
}

// One gene name against the positions of one chunk (lane lp, absolute p):
// sets the gene's bit when some lane holds a match.  WL: the name words are
// in LDS (wl) instead of global memory (gw); the two stay in separate code
// so that neither read becomes a flat load.
template <bool WL>
__device__ __forceinline__ void test_gene(const idb_gene_hdr &h, uint32_t g, const uint32_t *win, uint32_t w,
                                          uint32_t lp, uint32_t p, bool pv, uint32_t L, const uint32_t *wl,
                                          const uint32_t *gw, uint32_t *bits, uint32_t lane)
{
    if (h.len > L) return;  // longer than the row, or a name that never matches
    const uint32_t mask = h.len >= 4 ? 0xFFFFFFFFu : ((1u << (8 * h.len)) - 1u);
    bool ok = pv && p + h.len <= L && ((w ^ h.w0) & mask) == 0u;
    unsigned long long m = __ballot(ok);
    if (m && h.len > 4) {
        // the last 4 bytes
        if (ok) ok = win_word(win, lp + h.len - 4) == h.w1;
        m = __ballot(ok);
    }
    // the middle of the name, 4 bytes at a time
    for (uint32_t k = 4; m && k + 4 < h.len; k += 4) {
        const uint32_t gk = WL ? wl[h.woff + (k >> 2)] : gw[h.woff + (k >> 2)];
        if (ok) ok = win_word(win, lp + k) == gk;
        m = __ballot(ok);
    }
    if (m && lane == 0) bits[g >> 5] |= 1u << (g & 31);
}

template <bool WL>
__global__ __launch_bounds__(256) void k_gene_bitsets(const uint8_t *calls, const uint64_t *off, const uint32_t *len,
                                                      uint32_t n, const idb_gene_hdr *__restrict__ hdr,
                                                      const uint32_t *__restrict__ gw, uint32_t n_words,
                                                      uint32_t n_genes, int32_t *out, uint32_t width)
{
    __shared__ uint32_t win_all[GWPB][GWIN_WORDS];
    __shared__ uint32_t bits_all[GWPB][IDB_GENE_MAX_WIDTH];
    __shared__ idb_gene_hdr hl[GHDR_LDS];
    __shared__ uint32_t wl_all[GW_LDS];
    const uint32_t nl = n_genes < GHDR_LDS ? n_genes : GHDR_LDS;
    for (uint32_t g = threadIdx.x; g < nl; g += blockDim.x) hl[g] = hdr[g];
    if (WL)
        for (uint32_t k = threadIdx.x; k < n_words; k += blockDim.x) wl_all[k] = gw[k];
    __syncthreads();
    const uint32_t lane = __lane_id();
    const uint32_t wib = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint32_t *win = win_all[wib];
    uint32_t *bits = bits_all[wib];
    const uint32_t total = gridDim.x * GWPB;
    for (uint32_t row = blockIdx.x * GWPB + wib; row < n; row += total) {
        const uint32_t L = len[row];
        const uint8_t *src = calls + off[row];
        for (uint32_t k = lane; k < width; k += 64) bits[k] = 0u;
        for (uint32_t s0 = 0; s0 < L; s0 += GSEG) {
            // window bytes [s0, s0 + wl), zero past them
            const uint32_t wl = L - s0 < GWIN ? L - s0 : GWIN;
            const uint32_t nw = (wl + 3) / 4 + 2;
            for (uint32_t k = lane; k < nw; k += 64) {
                // four independent byte loads, each clamped into the row
                uint32_t v = 0u;
#pragma unroll
                for (uint32_t b = 0; b < 4; ++b) {
                    const uint32_t i = 4 * k + b;
                    const uint32_t c = src[s0 + (i < wl ? i : wl - 1)];
                    v |= (i < wl ? c : 0u) << (8 * b);
                }
                win[k] = v;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            const uint32_t pend = L - s0 < GSEG ? L - s0 : GSEG;  // start positions in this window
            for (uint32_t pc = 0; pc < pend; pc += 64) {
                const uint32_t lp = pc + lane;
                const bool pv = lp < pend;
                const uint32_t w = win_word(win, pv ? lp : 0u);
                const uint32_t p = s0 + lp;
                // headers from LDS, four at a time so that their reads overlap,
                // then (past the first GHDR_LDS) from global memory
                uint32_t g = 0;
                for (; g + 4 <= nl; g += 4) {
                    const idb_gene_hdr h0 = hl[g], h1 = hl[g + 1], h2 = hl[g + 2], h3 = hl[g + 3];
                    test_gene<WL>(h0, g, win, w, lp, p, pv, L, wl_all, gw, bits, lane);
                    test_gene<WL>(h1, g + 1, win, w, lp, p, pv, L, wl_all, gw, bits, lane);
                    test_gene<WL>(h2, g + 2, win, w, lp, p, pv, L, wl_all, gw, bits, lane);
                    test_gene<WL>(h3, g + 3, win, w, lp, p, pv, L, wl_all, gw, bits, lane);
                }
                for (; g < nl; ++g)
                    test_gene<WL>(hl[g], g, win, w, lp, p, pv, L, wl_all, gw, bits, lane);
                for (uint32_t g = nl; g < n_genes; ++g)
                    test_gene<WL>(hdr[g], g, win, w, lp, p, pv, L, wl_all, gw, bits, lane);
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        for (uint32_t k = lane; k < width; k += 64) out[(size_t)row * width + k] = (int32_t)bits[k];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    }
}

}  // namespace

hipError_t idb_launch_gene_bitsets(const uint8_t *calls, const uint64_t *off, const uint32_t *len, uint32_t n,
                                   const idb_gene_hdr *hdr, const uint32_t *gw, uint32_t n_words, uint32_t n_genes,
                                   int32_t *out, uint32_t width, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    if (width > IDB_GENE_MAX_WIDTH) return hipErrorInvalidValue;
    int per_cu = 0, dev = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)k_gene_bitsets<true>, 64 * GWPB, 0) !=
            hipSuccess ||
        per_cu <= 0)
        per_cu = 1;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
    (void)hipGetLastError();
    uint64_t blocks = ((uint64_t)n + GWPB - 1) / GWPB;
    const uint64_t cap = (uint64_t)per_cu * (uint64_t)cus;
    if (blocks > cap) blocks = cap;
    if (n_words <= GW_LDS)
        hipLaunchKernelGGL(k_gene_bitsets<true>, dim3((uint32_t)blocks), dim3(64 * GWPB), 0, s, calls, off, len, n,
                           hdr, gw, n_words, n_genes, out, width);
    else
        hipLaunchKernelGGL(k_gene_bitsets<false>, dim3((uint32_t)blocks), dim3(64 * GWPB), 0, s, calls, off, len, n,
                           hdr, gw, n_words, n_genes, out, width);
    return hipGetLastError();
}

uint32_t idb_gene_scan_blocks(uint32_t n, uint32_t threads, size_t lds)
{
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
    (void)hipGetLastError();
    // blocks that fit a CU by threads (2,048) and LDS (160 KB)
    const uint32_t fit = std::max<uint32_t>(1u, std::min<uint32_t>(2048u / threads, (uint32_t)(163840u / (lds + 512u))));
    return (uint32_t)std::min<uint64_t>(((uint64_t)n + threads - 1) / threads, (uint64_t)fit * cus);
}

// blob: the class map (256 bytes), the nodes, the table (16-bit entries when
// they go to LDS), each 16-byte aligned
hipError_t idb_launch_gene_scan(const uint8_t *calls, const uint64_t *off, const uint32_t *len, uint32_t n,
                                const uint8_t *cls, const uint32_t *nodes, const void *trans, bool narrow,
                                uint32_t ncls, uint32_t entries, uint32_t out_min, uint32_t n_nodes, uint32_t max_len,
                                int32_t *out, uint32_t width, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    const size_t lds = 256 + (narrow ? ((size_t)entries + 1) / 2 * 4 + 4 * (size_t)n_nodes : 0);
    // a bigger table shares one copy among more waves, so that a CU stays full
    const uint32_t threads = lds <= 19000 ? 256u : (lds <= 39000 ? 512u : 1024u);
    const dim3 grid(idb_gene_scan_blocks(n, threads, lds)), block(threads);
    const uint32_t wide = width == 4 && ((uintptr_t)out & 15u) == 0 ? 1u : 0u;
    // 16-bit tables of a few hundred names pass 64 KB (up to 82 KB: 32,768
    // entries and 4,096 nodes), which a kernel has to ask for
#define IDB_GS(TE, NW)                                                                                            \
    do {                                                                                                          \
        if (lds > 65536) {                                                                                        \
            const hipError_t e = hipFuncSetAttribute((const void *)k_gene_scan<TE, NW>,                           \
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);       \
            if (e != hipSuccess) return e;                                                                        \
        }                                                                                                         \
        hipLaunchKernelGGL((k_gene_scan<TE, NW>), grid, block, lds, s, calls, off, len, n, cls, (const TE *)trans, \
                           nodes, ncls, entries, out_min, n_nodes, max_len, out, width, wide);                    \
    } while (0)
    if (narrow) {
        if (width <= 4) IDB_GS(uint16_t, 4);
        else IDB_GS(uint16_t, 0);
    } else {
        if (width <= 4) IDB_GS(uint32_t, 4);
        else IDB_GS(uint32_t, 0);
    }
#undef IDB_GS
    return hipGetLastError();
}
