// idb_pairs_dev.h — device helpers shared by the pair kernels (idb_pairs.hip,
// idb_mx.hip): union-find, the gene gate, the per-wave staging of neighbour
// pairs, and the order in which waves take tiles.
#pragma once
#include "idb_internal.h"

namespace {

__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }

__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

__device__ __forceinline__ uint32_t rl(uint32_t v, uint32_t lane) { return __builtin_amdgcn_readlane(v, lane); }

__device__ __forceinline__ uint32_t ld_agent(const uint32_t *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ uint32_t uf_find(uint32_t *par, uint32_t x)
{
    uint32_t p = ld_agent(par + x);
    while (p != x) {
        const uint32_t gp = ld_agent(par + p);
        if (gp != p) {
            // path halving: gp is an ancestor of x, so the shortcut is safe
            __hip_atomic_store(par + x, gp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        x = p;
        p = gp;
    }
    return x;
}

// Link the larger root under the smaller one.  After a failed exchange the
// larger of the two roots strictly decreases, so the loop ends.
__device__ void uf_union(uint32_t *par, uint32_t a, uint32_t b)
{
    a = uf_find(par, a);
    b = uf_find(par, b);
    while (a != b) {
        if (a < b) {
            const uint32_t t = a;
            a = b;
            b = t;
        }
        uint32_t expected = a;
        if (__hip_atomic_compare_exchange_strong(par + a, &expected, b, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT))
            return;
        a = uf_find(par, expected);
        b = uf_find(par, b);
    }
}

__device__ __forceinline__ int lowest_common(const int32_t *a, const int32_t *b, uint32_t w)
{
    for (uint32_t k = 0; k < w; ++k) {
        const uint32_t m = (uint32_t)(a[k] & b[k]);
        if (m) return (int)(k * 32 + __builtin_ctz(m));
    }
    return -1;
}

// Exact canonical-bucket test from the bitsets (single-bucket mode: the V/J
// gate of cuda/BitsetVector.inl:214-237).
__device__ bool pair_in_bucket(const idb_pair_args &a, uint32_t x, uint32_t y, uint32_t bucket)
{
    const int32_t *vx = a.vbits + (size_t)x * a.vw, *vy = a.vbits + (size_t)y * a.vw;
    const int32_t *jx = a.jbits + (size_t)x * a.jw, *jy = a.jbits + (size_t)y * a.jw;
    const int lv = lowest_common(vx, vy, a.vw), lj = lowest_common(jx, jy, a.jw);
    if (a.single_bucket) return lv >= 0 && lj >= 0;
    return lv == (int)(bucket / a.gj) && lj == (int)(bucket % a.gj);
}

// The signature holds the residues mod 16 of the genes in question (canonical
// mode: genes below the bucket's; single-bucket mode: all genes).  Canonical
// mode: no common V residue and no common J residue -> no common lower gene ->
// canonical.  Single-bucket mode: no common V (or J) residue -> no common gene
// -> the gate fails.  Otherwise the bitsets decide.
__device__ __forceinline__ bool gate_pair(const idb_pair_args &a, bool chk_x, bool chk_y, uint32_t sx, uint32_t sy,
                                          uint32_t x, uint32_t y, uint32_t bucket)
{
    if (!(a.single_bucket || (chk_x && chk_y))) return true;
    const uint32_t c = sx & sy;
    if (a.single_bucket) {
        if ((c & 0xFFFFu) == 0u || (c >> 16) == 0u) return false;
    } else if (c == 0u) {
        return true;
    }
    return pair_in_bucket(a, x, y, bucket);
}

// Neighbour pairs are staged per wave in LDS (IDB_TILE entries) and appended
// to a chunk of the edge list that the wave owns; a new chunk costs one
// atomic on the chunk counter, so that counter sees one atomic per chunk
// instead of one per hit or per stage.  Past the capacity the counter keeps
// growing and the pairs are dropped, so the overflow is visible and the fuse
// pass over the tiles runs instead.
struct EdgeStage {
    uint2 *buf;       // this wave's IDB_TILE staging slots
    uint32_t n;       // staged pairs (wave-uniform)
    uint32_t chunk;   // the wave's current chunk, IDB_NONE before the first
    uint32_t fill;    // pairs written into it
};

// This block's copy of the run's statistics counters.
__device__ __forceinline__ unsigned long long *work_copy(const idb_pair_args &a)
{
    return a.work + IDB_WORK_U64 * (blockIdx.x & (IDB_WORK_COPIES - 1u));
}

// A wave's staging state.  The first chunk_base waves own the chunk of their
// number from the start: without that, every wave with a hit claims its first
// chunk from one counter, and thousands of waves' claims queue there (200k
// protein rows: the pass 156 -> 105 us, with one statistics atomic per block
// instead of per wave; the 2.6M-row batch's Hamming pass 517 -> 407 us).
__device__ __forceinline__ EdgeStage edge_stage(const idb_pair_args &a, uint2 *buf, uint32_t wave)
{
    return {buf, 0u, a.edges && wave < a.chunk_base ? wave : IDB_NONE, 0u};
}

// Adds the waves' statistics (lane 0's values) to the run's, one atomic per
// block and counter: sum holds N zeroed words of LDS.  All waves of the block
// come here.
template <int N>
__device__ __forceinline__ void add_stats(const idb_pair_args &a, unsigned long long *sum, const uint32_t (&slot)[N],
                                          const unsigned long long (&v)[N], uint32_t lane)
{
    if (lane == 0)
        for (int k = 0; k < N; ++k)
            if (v[k]) atomicAdd(sum + k, v[k]);
    __syncthreads();
    if (threadIdx.x == 0 && a.work)
        for (int k = 0; k < N; ++k)
            if (sum[k]) atomicAdd(work_copy(a) + slot[k], sum[k]);
}

__device__ __forceinline__ void close_chunk(const idb_pair_args &a, const EdgeStage &st, uint32_t lane)
{
    if (st.chunk != IDB_NONE && st.chunk < a.max_chunks && lane == 0) a.chunk_fill[st.chunk] = st.fill;
}

__device__ __forceinline__ void flush_edges(const idb_pair_args &a, EdgeStage &st, uint32_t lane)
{
    if (st.n == 0) return;
    if (st.chunk == IDB_NONE || st.fill + st.n > (1u << a.chunk_log2)) {
        close_chunk(a, st, lane);
        uint32_t c = 0;
        if (lane == 0) c = atomicAdd(a.n_chunks, 1u);
        st.chunk = __shfl(c, 0, 64);
        st.fill = 0;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    if (st.chunk < a.max_chunks && lane < st.n)
        a.edges[((size_t)st.chunk << a.chunk_log2) + st.fill + lane] = st.buf[lane];
    st.fill += st.n;
    st.n = 0;
}

__device__ __forceinline__ void stage_edges(const idb_pair_args &a, EdgeStage &st, bool keep, uint32_t x, uint32_t y,
                                            uint32_t lane)
{
    const unsigned long long km = __ballot(keep);
    if (!km || !a.edges) return;
    const uint32_t cnt = (uint32_t)__popcll(km);
    if (st.n + cnt > IDB_TILE) flush_edges(a, st, lane);
    if (keep) {
        const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(km >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)km, 0u));
        st.buf[st.n + below] = make_uint2(x, y);
    }
    st.n += cnt;
}

// End of a count-pass wave: last stage, last chunk's fill.
__device__ __forceinline__ void finish_edges(const idb_pair_args &a, EdgeStage &st, uint32_t lane)
{
    if (!a.edges) return;
    flush_edges(a, st, lane);
    close_chunk(a, st, lane);
}

// Fuse pass launched behind the union step without a host decision: it runs
// only when the pair list overflowed.
__device__ __forceinline__ bool fuse_skipped(const idb_pair_args &a)
{
    return a.fuse_if_overflow && *(volatile const uint32_t *)a.n_chunks <= a.max_chunks;
}

// The grid holds only as many waves as can be resident at once (no partly
// empty second round of waves trails the launch); wave w takes tiles w,
// w + waves, w + 2 waves, ...  A shared tile counter balances better in
// principle, but its device-scope atomics wait behind the pass's other
// atomics: measured on the 200k-row workload, claiming tiles (one counter per
// XCD, half of the tiles static) made the count pass slower, not faster.
__device__ __forceinline__ uint32_t next_tile(uint32_t ti, uint32_t total_waves) { return ti + total_waves; }

// The Myers count pass deals the rounds back and forth: wave w takes
// position w of even rounds and position waves - 1 - w of odd ones, so a wave
// that drew from a heavy stretch of one round draws from the other end of
// the next (3% off the 200k-row count pass).  n_tiles past the end.
__device__ __forceinline__ uint32_t step_tile(uint32_t ti, uint32_t total_waves, uint32_t n_tiles)
{
    if (ti >= n_tiles) return n_tiles;
    const uint32_t r = ti / total_waves, pos = ti % total_waves;
    const uint64_t nx = (uint64_t)(r + 1) * total_waves + (total_waves - 1 - pos);
    return nx < n_tiles ? (uint32_t)nx : n_tiles;
}

// Blocks are dealt to the 8 XCDs round-robin; renumber them so that each XCD
// starts on a contiguous run of tiles (neighbouring tiles share query blocks).
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t nb)
{
    const uint32_t per = nb / 8, rem = nb % 8, x = b % 8, k = b / 8;
    return x < rem ? x * (per + 1) + k : rem * (per + 1) + (x - rem) * per + k;
}

__device__ __forceinline__ int32_t t_of(uint32_t t2, bool fuse)
{
    return fuse ? (int32_t)(int16_t)(t2 >> 16) : (int32_t)(int16_t)(t2 & 0xFFFFu);
}

__device__ __forceinline__ idb_entry load_entry(const idb_entry *e)
{
    const uint4 *p = (const uint4 *)e;
    const uint4 a = p[0], b = p[1];
    idb_entry r;
    r.row = a.x;
    r.cp = a.y;
    r.len_chk = a.z;
    r.t2 = a.w;
    r.len = b.x;
    r.pres1 = b.y;
    r.pres2 = b.z;
    r.sig = b.w;
    return r;
}

// A tile record: the list is read-only during a pass and the index is
// wave-uniform, so this is a scalar load (waited on by lgkmcnt, which keeps
// it clear of the vector loads in flight).
__device__ __forceinline__ idb_tile tile_rec(const idb_pair_args &a, uint32_t ti)
{
    typedef const __attribute__((address_space(4))) uint32_t *const_words;
    const const_words w = (const_words)a.tiles + 4 * (size_t)ti;
    idb_tile t;
    t.q0 = w[0];
    t.t0 = w[1];
    t.bucket = w[2];
    t.shape = w[3];
    return t;
}

}  // namespace
