// idb_mx.hip — the count and fuse passes of fixed-threshold Levenshtein runs
// (t <= 3 edits on protein rows of up to 32 letters, t <= 4 on nucleotide
// rows), with the exact lower bound evaluated on the matrix cores.
//
// A wave owns a tile of up to 64 query x 64 target entries, as in
// idb_pairs.hip.  There the bound costs about 11 (letters) or 35 (3-grams)
// VALU instructions per query and lane, which is what the pass is bound by;
// here it is a 64 x 64 product of 4-bit feature vectors (mxfeat.h) on
// v_mfma_f32_32x32x64_f8f6f4, two products per pair (the bound in either
// direction), whose sign bits leave the accumulators with one OR and one
// shift-in per 64 pairs: 128 VALU instructions per tile.  Lane l then holds
// target l and a 64-bit mask of the queries that pass.  The length band is a
// mask too (one step per distinct query length of the tile), and so are the
// triangle of a diagonal tile and the canonical-bucket test.
//
// Pairs that pass are queued per wave and verified 64 at a time by the
// diagonal method on bit planes (lvdist.h): no per-tile Peq tables.  Protein
// rows keep their queue across tiles, so that batches are full, and read their
// 32-byte records from memory.  Nucleotide rows have ~260 such pairs a tile:
// the tile's records are staged in LDS (gathered from memory, 64 bytes per
// row and pair, the pass took 4.6 ms instead of 3.55 on 2M rows when it was
// written) and a first look at their substitutions decides most pairs.
// Measured (count kernel): 2M protein rows 9.28 -> 2.07 ms (320 VALU
// instructions per tile of 4,096 pairs, 1.7 ms of issue; the rest is the
// tiles' loads), 200k protein rows 0.225 -> 0.080 ms, 2M nucleotide rows of
// 24-154 letters 15.8 -> 3.17 ms (2.6 ms of VALU issue).
#include <algorithm>
#include <type_traits>

#include "idb_internal.h"
#include "idb_pairs_dev.h"
#include "lvdist.h"
#include "mxfeat.h"

namespace {

typedef int mx_i32x8 __attribute__((ext_vector_type(8)));
typedef uint32_t mx_u32x4 __attribute__((ext_vector_type(4)));
typedef float mx_f32x16 __attribute__((ext_vector_type(16)));

constexpr uint32_t MX_FP4 = 4;  // operand format code of E2M1

// NP planes of W words; KC feature chunks of 64 dimensions; threshold class T.
template <int NP_, int W_, int T_>
struct MxCfg {
    static constexpr int NP = NP_, W = W_, T = T_;
    static constexpr int KC = NP_ == 2 ? 3 : 1;
    static constexpr bool PER_TILE = NP_ == 2;             // records staged in LDS, queues emptied per tile
    // record words: planes, a spare word, copies, length in memory (protein rows);
    // planes, length, copies in LDS (nucleotide rows: an odd number of
    // 16-byte units, so that random records spread over the banks)
    static constexpr int VS = NP_ == 2 ? (W_ == 1 ? 4 : (W_ <= 5 ? 12 : 20)) : 8;
};

__device__ __forceinline__ mx_f32x16 mx_mul(const mx_u32x4 &a, const mx_u32x4 &b, const mx_f32x16 &c)
{
    const mx_i32x8 x = {(int)a.x, (int)a.y, (int)a.z, (int)a.w, 0, 0, 0, 0};
    const mx_i32x8 y = {(int)b.x, (int)b.y, (int)b.z, (int)b.w, 0, 0, 0, 0};
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x, y, c, MX_FP4, MX_FP4, 0, 0, 0, 0);
}

// Calls f(std::integral_constant<int, W'>) with the fewest words W' <= W that
// hold rows of lm letters (uniform over the wave).
template <int W, class F>
__device__ __forceinline__ void mx_words(uint32_t lm, F &&f)
{
    if (W > 2 && lm <= 64u) f(std::integral_constant<int, (W > 2 ? 2 : W)>{});
    else if (W > 3 && lm <= 96u) f(std::integral_constant<int, (W > 3 ? 3 : W)>{});
    else if (W > 4 && lm <= 128u) f(std::integral_constant<int, (W > 4 ? 4 : W)>{});
    else if (W > 5 && lm <= 160u) f(std::integral_constant<int, (W > 5 ? 5 : W)>{});
    else f(std::integral_constant<int, W>{});
}

// The records of one queued pair per lane (lanes < n): entries (e.x, e.y),
// read from memory or from the tile's records in LDS (rec: 64 queries from
// entry q0, then 64 targets from t0).
template <class G>
struct MxPair {
    uint32_t x[G::VS], y[G::VS];
    uint2 e;
    bool act;
    static constexpr int LEN = G::PER_TILE ? G::NP * G::W : G::NP * G::W + 2, CP = G::NP * G::W + 1;
    __device__ __forceinline__ MxPair(const idb_pair_args &a, const uint2 *queue, uint32_t n, uint32_t lane,
                                      const uint32_t *rec, uint32_t q0, uint32_t t0)
    {
        act = lane < n;
        e = queue[act ? lane : 0u];
        const mx_u32x4 *xp, *yp;
        if (G::PER_TILE) {
            xp = (const mx_u32x4 *)(rec + (e.x - q0) * G::VS);
            yp = (const mx_u32x4 *)(rec + (IDB_TILE + e.y - t0) * G::VS);
        } else {
            xp = (const mx_u32x4 *)(a.e_vrec + (size_t)e.x * G::VS);
            yp = (const mx_u32x4 *)(a.e_vrec + (size_t)e.y * G::VS);
        }
#pragma unroll
        for (int k = 0; k < G::VS / 4; ++k) {
            const mx_u32x4 u = xp[k], v = yp[k];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                x[4 * k + q] = u[q];
                y[4 * k + q] = v[q];
            }
        }
    }
    __device__ __forceinline__ int32_t lx() const { return (int32_t)x[LEN]; }
    __device__ __forceinline__ int32_t ly() const { return (int32_t)y[LEN]; }
};

// A pair found near: counts and the pair list, or (FUSE) the cluster forest.
// Counts go to the entries' counters (a row's are summed by k_mx_rows): the
// entries of a tile share a few lines, where their rows are scattered; with
// qacc, tacc (the counters of the tile's queries and targets from q0 and t0)
// a tile's counts are collected in LDS first.
template <class G, bool FUSE>
__device__ __forceinline__ void mx_near(const idb_pair_args &a, const MxPair<G> &p, bool hit, uint32_t lane,
                                        EdgeStage &est, uint32_t q0, uint32_t t0, int32_t *qacc, int32_t *tacc,
                                        unsigned long long &hits)
{
    if (!FUSE) {
        hits += __popcll(__ballot(hit));
        if (hit) {
            const int32_t cx = (int32_t)p.x[MxPair<G>::CP], cy = (int32_t)p.y[MxPair<G>::CP];
            if (G::PER_TILE) {
                atomicAdd(qacc + (p.e.x - q0), cy);
                atomicAdd(tacc + (p.e.y - t0), cx);
            } else {
                atomicAdd(a.cnt_e + p.e.x, cy);
                atomicAdd(a.cnt_e + p.e.y, cx);
            }
        }
        stage_edges(a, est, hit, p.e.x, p.e.y, lane);
    } else if (hit) {
        // (the gate let through pairs with at least one core row)
        const uint32_t rx = a.e_row[p.e.x], ry = a.e_row[p.e.y];
        const bool core_x = a.core[rx] != 0, core_y = a.core[ry] != 0;
        if (core_x && core_y) uf_union(a.par, rx, ry);
        else if (core_x) atomicMin(a.bmin + ry, rx);
        else if (core_y) atomicMin(a.bmin + rx, ry);
    }
}

// What a batch needs of its tile (nucleotide rows).
struct MxTile {
    const uint32_t *rec;          // the tile's records
    uint32_t q0, t0;
    int32_t *qacc, *tacc;
    uint32_t lm;                  // its longest row
};

// The exact decision for up to 64 queued pairs.
template <class G, bool FUSE>
__device__ __forceinline__ void mx_batch(const idb_pair_args &a, const MxTile &t, const uint2 *queue, uint32_t n,
                                         uint32_t lane, EdgeStage &est, unsigned long long &hits,
                                         unsigned long long &mlet)
{
    const MxPair<G> p(a, queue, n, lane, t.rec, t.q0, t.t0);
    if (!G::PER_TILE) mlet += p.act ? (uint32_t)p.lx() : 0u;
    bool near = false;
    mx_words<G::W>(t.lm, [&](auto w) {
        near = idb_lv_within<G::NP, decltype(w)::value, G::T, G::W>(p.x, p.y, p.lx(), p.ly(), a.t_const);
    });
    mx_near<G, FUSE>(a, p, p.act && near, lane, est, t.q0, t.t0, t.qacc, t.tacc, hits);
}

// Removes the first 64 of a queue's n entries.
__device__ __forceinline__ void mx_pop(uint2 *queue, uint32_t &n, uint32_t lane)
{
    const uint32_t rest = n - IDB_TILE;
    const uint2 moved = lane < rest ? queue[IDB_TILE + lane] : make_uint2(0u, 0u);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    if (lane < rest) queue[lane] = moved;
    n = rest;
}

// The first look at up to 64 of a tile's pairs: most pairs of nucleotide
// clones are of equal length and decided by their substitutions
// (idb_lv_equal_length); the others go to the second queue.
template <class G, bool FUSE>
__device__ __forceinline__ void mx_first(const idb_pair_args &a, const MxTile &t, const uint2 *queue, uint32_t n,
                                         uint32_t lane, EdgeStage &est, uint2 *queue2, uint32_t &n2,
                                         unsigned long long &hits, unsigned long long &mlet)
{
    {
        const MxPair<G> p(a, queue, n, lane, t.rec, t.q0, t.t0);
        mlet += p.act ? (uint32_t)p.lx() : 0u;
        int r = 2;
        mx_words<G::W>(t.lm, [&](auto w) {
            const int q = idb_lv_equal_length<G::NP, decltype(w)::value, G::T, G::W>(p.x, p.y, p.lx(), a.t_const);
            r = p.lx() == p.ly() ? q : 2;
        });
        if (!p.act) r = 0;
        mx_near<G, FUSE>(a, p, r == 1, lane, est, t.q0, t.t0, t.qacc, t.tacc, hits);
        const uint64_t um = __ballot(r == 2);
        if (r == 2) {
            const uint32_t below =
                __builtin_amdgcn_mbcnt_hi((uint32_t)(um >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)um, 0u));
            queue2[n2 + below] = p.e;
        }
        n2 += (uint32_t)__popcll(um);
    }
    if (n2 >= IDB_TILE) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        mx_batch<G, FUSE>(a, t, queue2, IDB_TILE, lane, est, hits, mlet);
        mx_pop(queue2, n2, lane);
    }
}

template <class G, bool FUSE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(G::W > 5 ? 2 : (G::NP == 2 ? 4 : 6)))) void k_mx(
    idb_pair_args a, uint32_t wpb)
{
    __shared__ uint2 queue_all[4][2 * IDB_TILE];
    __shared__ uint2 queue2_all[4][G::PER_TILE ? 2 * IDB_TILE : 1];
    __shared__ __align__(16) uint32_t rec_all[4][G::PER_TILE ? 2 * IDB_TILE * G::VS : 1];
    __shared__ uint2 edge_all[4][IDB_TILE];
    __shared__ int32_t acc_all[4][G::PER_TILE ? 2 * IDB_TILE : 1];
    const uint32_t lane = lane_id();
    const uint32_t wib = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (FUSE && fuse_skipped(a)) return;
    __shared__ unsigned long long stat_sum[5];
    if (threadIdx.x < 5) stat_sum[threadIdx.x] = 0;
    __syncthreads();
    uint2 *queue = queue_all[wib], *queue2 = queue2_all[wib];
    uint32_t qlen2 = 0;
    int32_t *qacc = acc_all[wib], *tacc = qacc + IDB_TILE;
    const uint32_t total_waves = gridDim.x * wpb;
    const uint32_t wave0 = (a.no_xcd_order ? blockIdx.x : xcd_block(blockIdx.x, gridDim.x)) + wib * gridDim.x;
    EdgeStage est = edge_stage(a, edge_all[wib], FUSE ? IDB_NONE : wave0);
    const int32_t t = a.t_const;
    const uint32_t h = lane >> 5, c = lane & 31u;
    // product row c of a 32-query half is query 16 h' + 4 g + e for
    // c = 8 g + 4 h' + e: the results' register r of lane half h is then
    // query 16 h + r
    const uint32_t qperm = 16u * ((c >> 2) & 1u) + 4u * (c >> 3) + (c & 3u);
    // the upper half-lanes' last word(s) carry the digits; on the other side
    // of each product stand the weights
    const uint32_t wmask = h ? (G::NP == 2 ? 0u : 0x0000FFFFu) : 0xFFFFFFFFu;
    const uint32_t wbits = h ? (G::NP == 2 ? IDB_MX_NT_WEIGHTS : IDB_MX_AA_WEIGHTS << 16) : 0u;
    const mx_u32x4 *feat = (const mx_u32x4 *)a.e_feat;
    const mx_f32x16 zero = {};
    unsigned long long gated = 0, hits = 0, mpairs = 0, mletters = 0, glane = 0, gllane = 0;
    uint32_t qlen = 0;
    // sub-tiles: a tile's queries in 2^sub_log2 parts (a part past the tile's
    // queries is empty)
    const uint32_t NT = a.n_tiles << a.sub_log2, part_n = IDB_TILE >> a.sub_log2;
    struct Part {
        uint32_t q0, t0, qn, tn, qoff;
        bool diag;
    };
    auto part_of = [&](uint32_t ti) {
        const idb_tile r = tile_rec(a, ti >> a.sub_log2);
        const uint32_t qoff = (ti & ((1u << a.sub_log2) - 1u)) * part_n;
        // signed: the compiler (ROCm 7.2) turns "qoff < n ? min(part_n, n -
        // qoff) : 0" on scalar registers into an unsigned difference that
        // does not stop at zero
        const int32_t rest = (int32_t)(r.shape & 0xFFu) - (int32_t)qoff;
        return Part{r.q0 + qoff, r.t0, (uint32_t)max(0, min((int32_t)part_n, rest)), (r.shape >> 8) & 0xFFu, qoff,
                    ((r.shape >> 16) & 1u) != 0u};
    };
    for (uint32_t ti = wave0; ti < NT; ti = step_tile(ti, total_waves, NT)) {
        const Part tile = part_of(ti);
        const uint32_t qn = tile.qn, tn = tile.tn, qoff = tile.qoff;
        const bool diag = tile.diag;
        if (!qn) continue;
        // features: rows past the tile's ends repeat its last entry (masked
        // below).  (Loading them one tile ahead cost more in registers than
        // it hid: 2.66 against 2.32 ms on 2M protein rows.)
        mx_u32x4 qf[2][G::KC], tf[2][G::KC];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const size_t qe = tile.q0 + min(32u * i + qperm, qn - 1u);
            const size_t te = tile.t0 + min(32u * i + c, tn - 1u);
#pragma unroll
            for (int k = 0; k < G::KC; ++k) {
                qf[i][k] = feat[(qe * G::KC + k) * 2 + h];
                tf[i][k] = feat[(te * G::KC + k) * 2 + h];
            }
        }
        const uint32_t mt = lane < tn ? a.e_meta[tile.t0 + lane] : 0u;
        const uint32_t mq = lane < qn ? a.e_meta[tile.q0 + lane] : 0u;
        const uint32_t m = mt & 0xFFFFu;
        // the bound: sign bits of both products (two 32-query halves i of
        // register r = query 32 i + 16 h + r, for targets c and c + 32)
        uint32_t fail[2] = {0u, 0u};
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if (32u * j >= tn) continue;
            mx_u32x4 tw = tf[j][G::KC - 1];
            tw.w = (tw.w & wmask) | wbits;
#pragma unroll
            for (int i = 1; i >= 0; --i) {
                // (a diagonal tile's later queries have no earlier targets)
                if (32u * i >= qn || (diag && qoff + 32u * i >= 32u * (j + 1))) {
                    fail[j] = fail[j] << 16;
                    continue;
                }
                mx_u32x4 qw = qf[i][G::KC - 1];
                qw.w = (qw.w & wmask) | wbits;
                mx_f32x16 s1 = zero, s2 = zero;
#pragma unroll
                for (int k = 0; k < G::KC; ++k) {
                    const bool last = k == G::KC - 1;
                    s1 = mx_mul(qf[i][k], last ? tw : tf[j][k], s1);
                    s2 = mx_mul(last ? qw : qf[i][k], tf[j][k], s2);
                }
#pragma unroll
                for (int r = 15; r >= 0; --r)
                    fail[j] = __builtin_amdgcn_alignbit(fail[j], __float_as_uint(s1[r]) | __float_as_uint(s2[r]), 31);
            }
        }
        // queries below this lane's limit (the upper triangle of a diagonal tile)
        const uint32_t dlim = lane >= tn ? 0u : (diag ? min(lane - min(lane, qoff), qn) : qn);
        // length band: one step per distinct query length
        uint32_t v0 = 0, v1 = 0;
        for (uint64_t rem = __ballot(lane < qn); rem;) {
            const uint32_t L = __builtin_amdgcn_readlane(mq, (uint32_t)__builtin_ctzll(rem)) & 0xFFFFu;
            const uint64_t same = __ballot(lane < qn && (mq & 0xFFFFu) == L);
            rem &= ~same;
            const bool in = (int32_t)__builtin_amdgcn_sad_u16(L, m, 0u) <= t;
            v0 |= in ? (uint32_t)same : 0u;
            v1 |= in ? (uint32_t)(same >> 32) : 0u;
        }
        v0 &= dlim >= 32u ? 0xFFFFFFFFu : (1u << dlim) - 1u;
        v1 &= dlim >= 64u ? 0xFFFFFFFFu : (dlim > 32u ? (1u << (dlim - 32u)) - 1u : 0u);
        // lane = target: its own bits for its half of the queries and the
        // other half-wave's for the other
        const auto sw = __builtin_amdgcn_permlane32_swap(fail[0], fail[1], false, false);
        const uint32_t fa = sw[0], fb = sw[1];  // queries 0..15 and 32..47; 16..31 and 48..63
        const uint32_t f0 = (fa & 0xFFFFu) | (fb << 16), f1 = (fa >> 16) | (fb & 0xFFFF0000u);
        // canonical bucket: pairs with a common gene below the bucket's belong to another one
        const uint64_t chkq = __ballot((mq >> 16) != 0u);
        if (chkq && __ballot((mt >> 16) != 0u)) {
            uint4 tl = make_uint4(0u, 0u, 0u, 0u), ql = tl;
            if (mt >> 16) tl = a.e_low[tile.t0 + lane];
            if (mq >> 16) ql = a.e_low[tile.q0 + lane];
            for (uint64_t cm = chkq; cm; cm &= cm - 1ull) {
                const uint32_t k = (uint32_t)__builtin_ctzll(cm);
                const uint32_t common = (__builtin_amdgcn_readlane(ql.x, k) & tl.x) |
                                        (__builtin_amdgcn_readlane(ql.y, k) & tl.y) |
                                        (__builtin_amdgcn_readlane(ql.z, k) & tl.z) |
                                        (__builtin_amdgcn_readlane(ql.w, k) & tl.w);
                if (common != 0u) {
                    if (k < 32u) v0 &= ~(1u << k);
                    else v1 &= ~(1u << (k - 32u));
                }
            }
        }
        if (FUSE) {
            // pairs with at least one core row
            const uint32_t rt = lane < tn ? a.e_row[tile.t0 + lane] : 0u;
            const uint32_t rq = lane < qn ? a.e_row[tile.q0 + lane] : 0u;
            const bool ct = lane < tn && a.core[rt] != 0;
            const uint64_t cq = __ballot(lane < qn && a.core[rq] != 0);
            v0 &= ct ? 0xFFFFFFFFu : (uint32_t)cq;
            v1 &= ct ? 0xFFFFFFFFu : (uint32_t)(cq >> 32);
        }
        const uint32_t gn = (uint32_t)(__builtin_popcount(v0) + __builtin_popcount(v1));
        glane += gn;
        gllane += (unsigned long long)gn * m;
        uint32_t p0 = v0 & ~f0, p1 = v1 & ~f1;
        MxTile mt_{rec_all[wib], tile.q0, tile.t0, qacc, tacc, 0u};
        if (G::PER_TILE) {
            if (!__ballot((p0 | p1) != 0u)) continue;
            // the tile's records: consecutive entries of each plane
            qacc[lane] = tacc[lane] = 0;
            uint32_t *rq = rec_all[wib] + lane * G::VS, *rt = rq + IDB_TILE * G::VS;
            const uint32_t *pq = a.e_vrec + tile.q0 + min(lane, qn - 1u), *pt = a.e_vrec + tile.t0 + min(lane, tn - 1u);
            constexpr int R = G::NP * G::W;
#pragma unroll
            for (int w = 0; w < R; ++w) {
                rq[w] = pq[(size_t)w * a.n_entries];
                rt[w] = pt[(size_t)w * a.n_entries];
            }
            rq[R] = mq & 0xFFFFu;
            rt[R] = m;
            rq[R + 1] = pq[(size_t)R * a.n_entries];
            rt[R + 1] = pt[(size_t)R * a.n_entries];
            // (entries are in length order)
            mt_.lm = max((uint32_t)__builtin_amdgcn_readlane(mq, qn - 1u) & 0xFFFFu,
                         (uint32_t)__builtin_amdgcn_readlane(mt, tn - 1u) & 0xFFFFu);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        }
        for (;;) {
            const uint64_t any = __ballot((p0 | p1) != 0u);
            if (!any) break;
            if (p0 | p1) {
                const uint32_t below =
                    __builtin_amdgcn_mbcnt_hi((uint32_t)(any >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)any, 0u));
                uint32_t k;
                if (p0) {
                    k = (uint32_t)__builtin_ctz(p0);
                    p0 &= p0 - 1u;
                } else {
                    k = 32u + (uint32_t)__builtin_ctz(p1);
                    p1 &= p1 - 1u;
                }
                queue[qlen + below] = make_uint2(tile.q0 + k, tile.t0 + lane);
            }
            const uint32_t np = (uint32_t)__popcll(any);
            qlen += np;
            mpairs += np;
            if (qlen >= IDB_TILE) {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                if (G::PER_TILE) mx_first<G, FUSE>(a, mt_, queue, IDB_TILE, lane, est, queue2, qlen2, hits, mletters);
                else mx_batch<G, FUSE>(a, mt_, queue, IDB_TILE, lane, est, hits, mletters);
                mx_pop(queue, qlen, lane);
            }
        }
        if (G::PER_TILE) {
            if (qlen) {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                mx_first<G, FUSE>(a, mt_, queue, qlen, lane, est, queue2, qlen2, hits, mletters);
                qlen = 0;
            }
            if (qlen2) {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                mx_batch<G, FUSE>(a, mt_, queue2, qlen2, lane, est, hits, mletters);
                qlen2 = 0;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        }
        if (G::PER_TILE && !FUSE) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            const int32_t qa = qacc[lane], ta = tacc[lane];
            if (qa) atomicAdd(a.cnt_e + tile.q0 + lane, qa);
            if (ta) atomicAdd(a.cnt_e + tile.t0 + lane, ta);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        }
    }
    if (!G::PER_TILE && qlen) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        mx_batch<G, FUSE>(a, MxTile{}, queue, qlen, lane, est, hits, mletters);
    }
    if (!FUSE) finish_edges(a, est, lane);
    mletters = wave_sum_u64(mletters);
    gated = wave_sum_u64(glane);
    const unsigned long long gletters = wave_sum_u64(gllane);
    if (FUSE) add_stats<1>(a, stat_sum, {2u}, {gated}, lane);
    else add_stats<5>(a, stat_sum, {0u, 1u, 3u, 5u, 6u}, {gated, hits, gletters, mpairs, mletters}, lane);
}

// Entry arrays of this pass, one thread per entry: the length for the tile
// builder, length and lower-gene flag (meta), features, record, lower genes,
// and the cluster growth's starting state.
template <int NP>
__global__ __launch_bounds__(256) void k_mx_fill(const uint64_t *ekey, const uint32_t *erow, uint32_t E,
                                                 const uint8_t *seq, uint32_t vw, uint32_t jw, uint32_t gj,
                                                 uint32_t gvj, const uint8_t *cmap, uint32_t K, uint32_t W, int32_t t,
                                                 uint32_t lb, uint16_t *elen, uint32_t *meta, uint32_t *feat,
                                                 uint32_t *vrec, uint8_t *bflag, uint32_t *inv, int32_t *cnt_e,
                                                 uint32_t *par_e, uint32_t *cmin_e, uint4 *elow, const uint4 *rrec)
{
    __shared__ uint8_t cm[256];
    for (uint32_t b = threadIdx.x; b < 256; b += blockDim.x) cm[b] = cmap[b];
    __syncthreads();
    for (uint32_t e = blockIdx.x * blockDim.x + threadIdx.x; e < E; e += gridDim.x * blockDim.x) {
        const uint64_t k = ekey[e];
        const uint32_t u = erow[e];
        const uint32_t L = (uint32_t)(k & ((1ull << lb) - 1ull));
        const uint64_t bucket = k >> lb;
        elen[e] = (uint16_t)L;
        par_e[e] = e;
        cmin_e[e] = IDB_NONE;
        cnt_e[e] = 0;
        bflag[e] = e == 0 || (ekey[e - 1] >> lb) != bucket;
        const uint32_t bl = (uint32_t)(bucket % gvj), gv = bl / gj, gjb = bl % gj;
        const uint4 r0 = rrec[2 * (size_t)u], r1 = rrec[2 * (size_t)u + 1];
        const uint32_t w[4] = {r1.x, r1.y, r1.z, r1.w};
        uint32_t lw[4], any = 0;
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
            const bool isv = q < vw, isj = q >= vw && q < vw + jw;
            lw[q] = isv || isj ? below_gene(w[q], isv ? q : q - vw, isv ? gv : gjb) : 0u;
            any |= lw[q];
        }
        elow[e] = make_uint4(lw[0], lw[1], lw[2], lw[3]);
        meta[e] = L | (any ? 0x10000u : 0u);
        // where the row lists its entries: in the order of its V, then J genes
        uint32_t vl = 0, jl = 0, nj = 0;
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
            if (q < vw) vl += __builtin_popcount(lw[q]);
            else if (q < vw + jw) {
                jl += __builtin_popcount(lw[q]);
                nj += __builtin_popcount(w[q]);
            }
        }
        inv[r0.w + vl * nj + jl] = e;
        const uint8_t *s = seq + ((uint64_t)r0.x | ((uint64_t)r0.y << 32));
        uint4 *f4 = (uint4 *)(feat + (size_t)e * (NP == 2 ? 24 : 8));
        if (NP == 5) {
            // at most 32 letters, codes below 30: five planes of one word
            uint32_t pl[5] = {0u, 0u, 0u, 0u, 0u}, b1 = 0, b2 = 0;
            for (uint32_t k0 = 0; k0 < L; k0 += 16) {
                const uint4 v = row16(s, L, k0);
#pragma unroll
                for (uint32_t b = 0; b < 16; ++b) {
                    const uint32_t code = cm[byte_of(v, b)];
                    if (k0 + b < L) {
                        const uint32_t bit = 1u << code;
                        b2 |= b1 & bit;
                        b1 |= bit;
#pragma unroll
                        for (uint32_t p = 0; p < 5; ++p) pl[p] |= ((code >> p) & 1u) << (k0 + b);
                    }
                }
            }
            uint64_t f = (uint64_t)b1 | ((uint64_t)b2 << K);
            const int32_t n = __builtin_popcount(b1) + __builtin_popcount(b2);
            uint32_t d[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) d[q] = idb_mx_spread((uint32_t)(f >> (8 * q)));
            d[7] |= idb_mx_digits(t - n, 2) << 16;
            f4[0] = make_uint4(d[0], d[1], d[2], d[3]);
            f4[1] = make_uint4(d[4], d[5], d[6], d[7]);
            uint4 *r4 = (uint4 *)(vrec + (size_t)e * 8);
            r4[0] = make_uint4(pl[0], pl[1], pl[2], pl[3]);
            r4[1] = make_uint4(pl[4], 0u, r0.z, L);
        } else {
            uint32_t g[6] = {0u, 0u, 0u, 0u, 0u, 0u}, hist = 0;
            for (uint32_t wd = 0; wd < W; ++wd) {
                uint32_t a0 = 0, a1 = 0;
                for (uint32_t k0 = 32 * wd; k0 < 32 * wd + 32 && k0 < L; k0 += 16) {
                    const uint4 v = row16(s, L, k0);
                    // (all 16 letters, those past the row's end masked: the
                    // letter map's LDS reads then run ahead of the profile)
                    const uint32_t nb = min(16u, L - k0);
                    uint32_t code[16], p0 = 0, p1 = 0;
#pragma unroll
                    for (uint32_t b = 0; b < 16; ++b) code[b] = cm[byte_of(v, b)] & 3u;
#pragma unroll
                    for (uint32_t b = 0; b < 16; ++b) {
                        p0 |= (code[b] & 1u) << b;
                        p1 |= (code[b] >> 1) << b;
                        hist = ((hist << 2) | code[b]) & 63u;
                        if (b < nb && k0 + b >= 2) idb_qmask_add(g, hist);
                    }
                    const uint32_t in = (1u << nb) - 1u;
                    a0 |= (p0 & in) << (k0 & 31u);
                    a1 |= (p1 & in) << (k0 & 31u);
                }
                vrec[(size_t)wd * E + e] = a0;
                vrec[(size_t)(W + wd) * E + e] = a1;
            }
            vrec[(size_t)(2 * W) * E + e] = r0.z;
            g[5] &= IDB_MX_NT_L3HI;
            int32_t n = 0;
#pragma unroll
            for (int q = 0; q < 6; ++q) n += __builtin_popcount(g[q]);
#pragma unroll
            for (int q = 0; q < 6; ++q) {
                uint32_t d[4];
#pragma unroll
                for (int b = 0; b < 4; ++b) d[b] = idb_mx_spread(g[q] >> (8 * b));
                if (q == 5) d[3] = idb_mx_digits(3 * t - n, 6);
                f4[q] = make_uint4(d[0], d[1], d[2], d[3]);
            }
        }
    }
}

// Rows after the count pass: a unique row's count is its copies plus its
// entries' counts; its core flag goes to the row and to its entries, which
// are linked into one component for the cluster growth (the first one stands
// for the row).  Duplicate rows count 0 (core only when min_pts is 0).
__global__ __launch_bounds__(256) void k_mx_rows(const uint32_t *uniq, const uint32_t *num, const uint64_t *eoff,
                                                 const uint32_t *inv, const int32_t *cnt_e, const uint32_t *copies,
                                                 uint32_t n, int32_t minpts, int32_t *cnt, int32_t *core, uint32_t *pe,
                                                 uint8_t *ecore, uint32_t *par_e, uint32_t *n_cores,
                                                 unsigned long long *stamps)
{
    idb_stamp_start(stamps + IDB_T_COUNT);
    __shared__ uint32_t part[4];
    const uint32_t U = num[0], step = gridDim.x * blockDim.x, i0 = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t local = 0;
    for (uint32_t k = i0; k < U; k += step) {
        const uint32_t u = uniq[k], a = (uint32_t)eoff[k], b = (uint32_t)eoff[k + 1];
        const uint32_t first = a < b ? inv[a] : IDB_NONE;
        int32_t c = (int32_t)copies[u];
        for (uint32_t i = a; i < b; ++i) c += cnt_e[i == a ? first : inv[i]];
        const bool is = c >= minpts;
        cnt[u] = c;
        core[u] = is;
        local += is;
        if (a < b) {
            pe[u] = first | (is ? 0x80000000u : 0u);
            for (uint32_t i = a; i < b; ++i) {
                const uint32_t e = i == a ? first : inv[i];
                ecore[e] = is;
                if (is && i > a) {
                    const uint32_t lo = e < first ? e : first, hi = e < first ? first : e;
                    atomicMin(par_e + hi, lo);
                }
            }
        }
    }
    const bool dup_core = 0 >= minpts;
    for (uint32_t i = i0; i < n; i += step)
        if (copies[i] == 0u) {
            core[i] = dup_core;
            local += dup_core;
        }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) local += (uint32_t)__shfl_xor((int)local, o, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = local;
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t t = part[0] + part[1] + part[2] + part[3];
        if (t) atomicAdd(n_cores + (blockIdx.x & 15u), t);  // 16 counters
    }
    idb_stamp_end(stamps + IDB_T_CORE);
}

template <class G, bool FUSE>
hipError_t launch_mx_g(const idb_pair_args &a_in, hipStream_t s)
{
    idb_pair_args a = a_in;
    const bool tuned = a.tune_wpb != 0 || a.tune_grid_mul != 0;
    const uint32_t wpb = tuned ? idb_pick_wpb(a, 4) : 4u;
    const void *k = (const void *)k_mx<G, FUSE>;
    const uint32_t resident = idb_resident_blocks(k, 64 * wpb, 0);
    // Launch shape, measured (count kernel).  Grid: 8x the resident blocks once
    // a wave has 16 tiles (2M protein rows 2.20 -> 2.08 ms, 2M nucleotide rows
    // 3.90 -> 3.55 ms when it was set), else 2x (200k protein rows 0.083 against
    // 0.107 ms at 4x).  Few tiles are taken in 2 or 4 parts each, while the parts fit
    // half the resident waves (protein rows: 442 tiles 33 -> 17 us, 1,202
    // tiles 32 -> 25 us in 2 parts but 33 us in 4) or twice of them
    // (nucleotide rows, whose batches are longer: 471 tiles 69 -> 32 us,
    // 2,586 tiles 110 -> 68 us).
    if (!tuned) {
        a.no_xcd_order = 1;
        a.tune_grid_mul = a.n_tiles >= 16ull * resident * wpb ? 8u : 2u;
    }
    const uint64_t fit = G::PER_TILE ? 2ull * resident * wpb : (uint64_t)resident * wpb / 2;
    a.sub_log2 = 4ull * a.n_tiles <= fit ? 2u : (2ull * a.n_tiles <= fit ? 1u : 0u);
    const dim3 block(64 * wpb),
        grid(FUSE ? idb_grid_for(a.n_tiles << a.sub_log2, wpb, resident, a.tune_grid_mul)
                  : idb_count_grid(a, a.n_tiles << a.sub_log2, wpb, resident));
    hipLaunchKernelGGL((k_mx<G, FUSE>), grid, block, 0, s, a, wpb);
    return hipGetLastError();
}

template <int NP, int W, bool FUSE>
hipError_t launch_mx_w(const idb_pair_args &a, hipStream_t s)
{
    if (a.t_const <= 1) return launch_mx_g<MxCfg<NP, W, 1>, FUSE>(a, s);
    if (a.t_const == 2) return launch_mx_g<MxCfg<NP, W, 2>, FUSE>(a, s);
    if (a.t_const == 3) return launch_mx_g<MxCfg<NP, W, 3>, FUSE>(a, s);
    if (NP == 2 && a.t_const == 4) return launch_mx_g<MxCfg<NP, W, NP == 2 ? 4 : 3>, FUSE>(a, s);
    return hipErrorInvalidValue;
}

template <bool FUSE>
hipError_t launch_mx(const idb_pair_args &a, hipStream_t s)
{
    if (a.n_tiles == 0) return hipSuccess;
    if (a.mx_planes == 5 && a.mx_words == 1) return launch_mx_w<5, 1, FUSE>(a, s);
    if (a.mx_planes == 2) switch (a.mx_words) {
        case 1: return launch_mx_w<2, 1, FUSE>(a, s);
        case 2: return launch_mx_w<2, 2, FUSE>(a, s);
        case 3: return launch_mx_w<2, 3, FUSE>(a, s);
        case 5: return launch_mx_w<2, 5, FUSE>(a, s);
        case 8: return launch_mx_w<2, 8, FUSE>(a, s);
        default: break;
        }
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t idb_launch_mx_count(const idb_pair_args &a, hipStream_t s) { return launch_mx<false>(a, s); }
hipError_t idb_launch_mx_fuse(const idb_pair_args &a, hipStream_t s) { return launch_mx<true>(a, s); }

hipError_t idb_launch_mx_rows(const idb_mx_rows_args &r, hipStream_t s)
{
    const uint32_t blocks = std::max<uint32_t>(1u, std::min<uint32_t>((r.n + 255u) / 256u, 2048u));
    hipLaunchKernelGGL(k_mx_rows, dim3(blocks), dim3(256), 0, s, r.uniq, r.num, r.eoff, r.inv, r.cnt_e, r.copies, r.n,
                       r.min_pts, r.cnt, r.core, r.pe, r.ecore, r.par_e, r.n_cores, r.stamps);
    return hipGetLastError();
}

hipError_t idb_launch_mx_fill(const idb_mx_fill_args &f, hipStream_t s)
{
    const uint32_t blocks = std::max<uint32_t>(1u, std::min<uint32_t>((f.E + 255u) / 256u, 2048u));
    if (f.planes == 5)
        hipLaunchKernelGGL(k_mx_fill<5>, dim3(blocks), dim3(256), 0, s, f.ekey, f.erow, f.E, f.seq, f.vw, f.jw, f.gj,
                           f.gvj, f.cmap, f.K, f.W, f.t, f.lb, f.elen, f.meta, f.feat, f.vrec, f.bflag, f.inv, f.cnt_e,
                           f.par_e, f.cmin_e, f.elow, f.rrec);
    else
        hipLaunchKernelGGL(k_mx_fill<2>, dim3(blocks), dim3(256), 0, s, f.ekey, f.erow, f.E, f.seq, f.vw, f.jw, f.gj,
                           f.gvj, f.cmap, f.K, f.W, f.t, f.lb, f.elen, f.meta, f.feat, f.vrec, f.bflag, f.inv, f.cnt_e,
                           f.par_e, f.cmin_e, f.elow, f.rrec);
    return hipGetLastError();
}
