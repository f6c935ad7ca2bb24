// idb_learned.hip — the learned candidate filter's encoder on gfx950: a small
// 1-D CNN over CDR3 letters, trained and run by this file's own kernels.
//
// No counterpart in the reference (it evaluates every pair exactly).  The
// encoder maps a row to a unit vector z; the learned filter proposes the pairs
// of a tile whose dot product z_x . z_y reaches a threshold, and the exact
// Myers kernel verifies every proposal, so distances are never approximated.
//
//   tokens (<= P letters) -> embedding 32 x 32 -> 3 x [conv1d k=5 'same',
//   128 channels, GELU] -> mean over letters -> linear 128 -> 64 -> L2 norm.
//
// P, the positions per row, is fixed when the encoder is made: 32 for
// protein rows, 160 for nucleotide rows of up to 160 letters.
//
// Weights are bfloat16 copies of float32 master weights (Adam keeps the
// master copy); activations are bfloat16, all products accumulate in float32.
// Rows are packed back to back with two zero rows after each (the zero
// padding of a 5-tap window), in tiles of 256.  One fused kernel (k_encode)
// runs the forward pass of a tile in LDS, a second one (k_enc_bwd) the data
// gradients; only what the weight gradients (k_wgrad) read goes through HBM.
// All products run on v_mfma_f32_32x32x16_bf16.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <random>
#include <string>
#include <vector>

#include "copy_pool.h"
#include "idb_internal.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t T = 5, NTOK = 32, C0 = 32, C = 128, D = 64;
constexpr float GELU_K = 0.7978845608028654f;  // sqrt(2 / pi)

// Flat parameter layout (float32 master and bfloat16 copy share it).
constexpr uint32_t O_EMB = 0, O_W1 = O_EMB + NTOK * C0, O_B1 = O_W1 + C * T * C0, O_W2 = O_B1 + C,
                   O_B2 = O_W2 + C * T * C, O_W3 = O_B2 + C, O_B3 = O_W3 + C * T * C, O_WP = O_B3 + C,
                   O_BP = O_WP + D * C, N_PARAMS = O_BP + D;
static_assert(N_PARAMS == IDB_ENC_PARAMS, "parameter count");

// Round to nearest even (the hardware conversion, one instruction).
__device__ __forceinline__ uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// 0.5 x (1 + tanh(u)) = x / (1 + exp(-2u)), u = k (x + 0.044715 x^3): one
// hardware base-2 exponential and one reciprocal.  For very negative x the
// exponential overflows to inf and the result is -0; for large x it is x.
__device__ __forceinline__ float gelu(float x)
{
    constexpr float C1 = -2.f * GELU_K * 1.4426950408889634f, C3 = C1 * 0.044715f;  // -2u log2(e) = x (C1 + C3 x^2)
    const float e = x * __builtin_fmaf(C3, x * x, C1);
    return x * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(e));
}
// Its derivative s + x s (1 - s) d(2u)/dx with s = 1 / (1 + exp(-2u)).
__device__ __forceinline__ float gelu_grad(float x)
{
    constexpr float C1 = -2.f * GELU_K * 1.4426950408889634f, C3 = C1 * 0.044715f;
    const float x2 = x * x;
    const float s = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(x * __builtin_fmaf(C3, x2, C1)));
    const float du2 = __builtin_fmaf(6.f * GELU_K * 0.044715f, x2, 2.f * GELU_K);
    return s + x * du2 * (s - s * s);
}

__global__ void k_to_bf16(const float *src, uint32_t n, uint16_t *dst)
{
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) dst[i] = f2bf(src[i]);
}

__global__ void k_adam(float *th, const float *g, float *m, float *v, uint32_t n, float lr, float b1, float b2,
                       float eps, float c1, float c2, uint16_t *thb)
{
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.f - b1) * gi;
        const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        const float t = th[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
        th[i] = t;
        thb[i] = f2bf(t);
    }
}

// ---------------------------------------------------------------------------
// The whole forward pass in one kernel.
//
// A block takes a tile of EM = 64 RT activation rows (256 or 128) and keeps them in LDS
// through all three convolutions (layer by layer, in place), so neither
// activations nor im2col windows touch HBM.  Sequences are packed back to
// back with two zero rows between them: a 5-tap window reaches two rows, so
// that is the zero padding of both neighbours, and no row is spent on
// positions past a sequence's end (protein rows average 15 of 32 positions,
// 24-150-letter rows 87 of 160).  Products run transposed (channels x rows):
// a lane then holds four consecutive channels of one row, which leave as one
// 8-byte LDS store, and validity is one bit per lane.
//   4 waves of 64 channels x 128 rows: per 16-deep k step 8 MFMAs (256
// cycles) take 4 row fragments from LDS (50% of its bandwidth over the 4
// waves) and 2 weight fragments from L2, packed so that a wave reads 1 KB
// in a row.  128 accumulators leave room for 2 waves per SIMD; at 71 KB of
// activations two blocks share a CU, so one block's GELU overlaps the other's
// products (200k protein rows: 388M VALU instructions, 632 us of issue, beside
// 513 us of MFMAs).
// In training (TRAIN) a block also writes what the backward pass reads: the
// pre-activations in the lanes' own order (512 bytes per wave and store; k_enc_bwd
// has the same lane mapping), the layers' inputs row by row in packed order,
// the pooled means and the norms.
// Measured: 200k protein rows (1.29 Tflop of MFMAs) 5.22 -> 1.60 ms, 806 TFLOP/s
// (a large bf16 product reaches 1,205 here); 20k rows of 24-150 letters in the
// five segments of an embedding call 2.98 -> 1.07 ms.
constexpr uint32_t EST = C + 8;                   // LDS row stride (272 bytes: conflict-free)
constexpr uint32_t EPW = 1024;                    // sequences per packing window
constexpr uint32_t EGRP = 8;                      // sequences per round of the head
constexpr uint32_t EKS1 = T * C0 / 16, EKS = T * C / 16;  // k steps of layer 1, of layers 2 and 3
constexpr size_t EPACK = (size_t)(EKS1 + 2 * EKS) * 4 * 64 * 8;  // packed weights (bfloat16)
constexpr uint32_t BLAYER = EKS * 4 * 64 * 8, BPACK = 2 * BLAYER + EKS * 64 * 8;  // and transposed
constexpr uint32_t EPAD = 4 * 2048;               // fragments loaded ahead past a pack's end

// Where a training batch's sequences come from: sequence 2 i + h is row
// pairs[2 q + h] of pair q = order[first + i] (or first + i).
struct PairSource {
    const uint32_t *pairs, *order;
    const float *labels;
    uint64_t first;
    uint32_t *rows, *blen;  // out: row and length of every sequence
    float *y;               // out: label of every pair
};

// A tile: first sequence, sequences, first row in packed order, packed rows.
// Greedy packing of consecutive sequences into tiles, window by window:
// tiles in any order, and every sequence's first row within its tile.  At
// most EM + 2 rows per tile counting each sequence's two zero rows (the last
// two lie in the tile's zero border).  Segments of wseg windows keep their
// tiles from the place of their first sequence on: count[2 s] = tiles of
// segment s, count[1] = packed rows (training, one segment).
template <bool TRAIN>
__global__ __launch_bounds__(256) void k_enc_plan(const uint32_t *len, uint32_t n, uint32_t P, uint32_t em, uint32_t wseg, uint4 *tiles,
                                                  uint32_t *count, uint16_t *rstart, PairSource ps)
{
    __shared__ uint32_t S[EPW + 1], cut[EPW + 1], part[4], base_s, base_r;
    __shared__ uint16_t nxt[EPW];
    const uint32_t w0 = blockIdx.x * EPW, m = min(EPW, n - w0), tid = threadIdx.x, lane = tid & 63;
    constexpr uint32_t PER = EPW / 256;
    uint32_t v[PER], sum = 0;
#pragma unroll
    for (uint32_t k = 0; k < PER; ++k) {
        const uint32_t i = tid * PER + k;
        v[k] = 0u;
        if (i < m) {
            uint32_t L;
            if (TRAIN) {
                const uint32_t b = w0 + i;
                const uint64_t at = ps.first + (b >> 1);
                const uint32_t q = ps.order ? ps.order[at] : (uint32_t)at;
                const uint32_t r = ps.pairs[2 * (size_t)q + (b & 1u)];
                L = min(len[r], P);
                ps.rows[b] = r;
                ps.blen[b] = L;
                if ((b & 1u) == 0) ps.y[b >> 1] = ps.labels[q];
            } else {
                L = min(len[w0 + i], P);
            }
            v[k] = L + 2u;
        }
        sum += v[k];
    }
    uint32_t inc = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = (uint32_t)__shfl_up((int)inc, o, 64);
        if (lane >= (uint32_t)o) inc += t;
    }
    if (lane == 63) part[tid >> 6] = inc;
    __syncthreads();
    uint32_t at = inc - sum;
    for (uint32_t w = 0; w < (tid >> 6); ++w) at += part[w];
#pragma unroll
    for (uint32_t k = 0; k < PER; ++k) {
        S[tid * PER + k] = at;
        at += v[k];
    }
    if (tid == 255) S[EPW] = at;
    __syncthreads();
    // the tile that starts at sequence i ends before nxt[i]
    for (uint32_t i = tid; i < m; i += 256) {
        uint32_t lo = i + 1, hi = m;  // S[lo] - S[i] fits (one sequence always does)
        while (lo < hi) {
            const uint32_t mid = (lo + hi + 1) >> 1;
            if (S[mid] - S[i] <= em + 2u) lo = mid; else hi = mid - 1;
        }
        nxt[i] = (uint16_t)lo;
    }
    __syncthreads();
    if (tid == 0) {
        uint32_t c = 0;
        for (uint32_t i = 0; i < m; i = nxt[i]) cut[c++] = i;
        cut[c] = m;
        part[0] = c;
        const uint32_t seg = blockIdx.x / wseg;
        base_s = seg * wseg * EPW + atomicAdd(count + 2 * seg, c);
        base_r = TRAIN ? atomicAdd(count + 1, S[m]) : 0u;
    }
    __syncthreads();
    const uint32_t c = part[0];
    for (uint32_t t = tid; t < c; t += 256)
        tiles[base_s + t] = make_uint4(w0 + cut[t], cut[t + 1] - cut[t], base_r + S[cut[t]], S[cut[t + 1]] - S[cut[t]]);
    for (uint32_t i = tid; i < m; i += 256) {
        uint32_t lo = 0, hi = c;  // last tile that starts at or before i
        while (lo + 1 < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (cut[mid] <= i) lo = mid; else hi = mid;
        }
        rstart[w0 + i] = (uint16_t)(S[i] - S[cut[lo]]);
    }
}

// Weights in the order the encoder's waves read them: per layer and k step,
// four 32-channel fragments of 64 lanes x 8 values; then the projection as
// (input pair, output) words and as (output, input pair) words; then, for the
// data gradients, layers 3 and 2 transposed (40 k steps of four fragments
// each) and layer 1 (40 k steps of one fragment).
__global__ void k_enc_pack(const uint16_t *theta_b, uint16_t *dst, uint32_t *wp2, uint16_t *bdst)
{
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < EPACK; i += gridDim.x * blockDim.x) {
        const uint32_t e = i & 7u, ln = (i >> 3) & 63u, ct = (i >> 9) & 3u;
        uint32_t ks = i >> 11, cin = C0, o = O_W1;
        if (ks >= EKS1) {
            ks -= EKS1;
            cin = C;
            o = O_W2;
            if (ks >= EKS) {
                ks -= EKS;
                o = O_W3;
            }
        }
        dst[i] = theta_b[o + (ct * 32 + (ln & 31u)) * (T * cin) + ks * 16 + (ln >> 5) * 8 + e];
    }
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < C / 2 * D; i += gridDim.x * blockDim.x) {
        const uint32_t d = i % D, o = 2 * (i / D);
        wp2[i] = (uint32_t)theta_b[O_WP + d * C + o] | ((uint32_t)theta_b[O_WP + d * C + o + 1] << 16);
    }
    // k step ks of a transposed layer: tap ks / 8, output channels 16 (ks % 8) ..
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < BPACK; i += gridDim.x * blockDim.x) {
        const uint32_t e = i & 7u, ln = (i >> 3) & 63u;
        const bool l1 = i >= 2 * BLAYER;
        const uint32_t at = (l1 ? i - 2 * BLAYER : i % BLAYER) >> 9, ct = l1 ? 0u : at & 3u, ks = l1 ? at : at >> 2;
        const uint32_t cin = l1 ? C0 : C, w = l1 ? O_W1 : (i < BLAYER ? O_W3 : O_W2);
        const uint32_t o = (ks & 7u) * 16 + (ln >> 5) * 8 + e, c = ct * 32 + (ln & 31u);
        bdst[i] = theta_b[w + o * (T * cin) + (ks >> 3) * cin + c];
    }
}

// Rows of a tile: 64 RT.  Embedding takes 256 (RT = 4): two blocks a CU, and
// the least padding (200k protein rows 1.58 ms, tiles of 128 rows 1.63).  A
// training batch is a few tiles per CU, so that the spread of the tiles over
// the CUs and the latency of one tile count: 128 rows (three blocks a CU)
// where P fits, 4,096 protein pairs forward 135 -> 105 us, backward 204 ->
// 157, 256 pairs 54 -> 39 and 84 -> 55.
constexpr int enc_blocks_per_cu(int rt) { return rt == 4 ? 2 : 3; }

struct EncArgs {
    const uint8_t *seq;
    const uint64_t *off;
    const uint32_t *len;
    const uint4 *tiles;
    const uint32_t *n_tiles;
    const uint16_t *rstart;
    const uint8_t *vocab;
    const uint16_t *theta_b, *pack;
    const uint32_t *wp2;
    uint32_t P;
    float *z;        // either may be null
    uint16_t *zb;
    // training
    const uint32_t *rows;  // row of each sequence (len is per sequence)
    uint2 *H[3];           // pre-activations, lane order: 8192 words of 8 bytes per tile
    uint16_t *X0, *A1, *A2;
    float *pool, *nrm;
};

// One convolution over the tile: acc = W x window, CIN input channels.  REV:
// taps in the order of the data gradient (window row 4 - t for tap t).
template <uint32_t CIN, int RT, bool REV = false>
__device__ __forceinline__ void enc_conv(const uint16_t *X, const u32x4 *wp, uint32_t lane, f32x16 (&acc)[2][RT])
{
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < RT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    // k steps per tap; steps of weight fragments loaded ahead (four against
    // two measured the same, 1.58 ms for 200k protein rows)
    constexpr uint32_t KT = CIN / 16, AHEAD = CIN == C0 ? 2 : 4;
    const uint16_t *xr = X + (lane & 31u) * EST + (lane >> 5) * 8;
    u32x4 wq[AHEAD][2];
#pragma unroll
    for (uint32_t a = 0; a < AHEAD; ++a) {
        wq[a][0] = wp[a * 256 + lane];
        wq[a][1] = wp[a * 256 + 64 + lane];
    }
#pragma unroll 1
    for (uint32_t t = 0; t < T; ++t) {
        const uint16_t *xt = xr + (REV ? T - 1 - t : t) * EST;
        const u32x4 *wt = wp + t * KT * 256;
#pragma unroll
        for (uint32_t c = 0; c < KT; ++c) {
            bf16x8 w0 = __builtin_bit_cast(bf16x8, wq[c % AHEAD][0]), w1 = __builtin_bit_cast(bf16x8, wq[c % AHEAD][1]);
            // (past the layer's last step: the next layer's first fragments,
            // or the buffer's padding)
            wq[c % AHEAD][0] = wt[(c + AHEAD) * 256 + lane];
            wq[c % AHEAD][1] = wt[(c + AHEAD) * 256 + 64 + lane];
#pragma unroll
            for (int j = 0; j < RT; ++j) {
                const bf16x8 x = *(const bf16x8 *)(xt + j * 32 * EST + c * 16);
                acc[0][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w0, x, acc[0][j], 0, 0, 0);
                acc[1][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w1, x, acc[1][j], 0, 0, 0);
            }
        }
    }
}

// Rows [0, used) of the tile in LDS (its zero border included), to packed rows.
__device__ __forceinline__ void enc_store_rows(const uint16_t *X, uint16_t *out, uint32_t used, uint32_t tid)
{
    for (uint32_t r = tid >> 4; r < used; r += 16)
        *(u32x4 *)(out + (size_t)r * C + (tid & 15u) * 8) = *(const u32x4 *)(X + (r + 2) * EST + (tid & 15u) * 8);
}

// Index of the sequence that row r of a tile belongs to.
__device__ __forceinline__ uint32_t seq_of_row(const uint16_t *s_row, uint32_t cnt, uint32_t r)
{
    uint32_t lo = 0, hi = cnt;
    while (lo + 1 < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (s_row[mid] <= r) lo = mid; else hi = mid;
    }
    return lo;
}

template <bool TRAIN, int RT>
__global__ __launch_bounds__(256, enc_blocks_per_cu(RT)) void k_encode(EncArgs a)
{
    constexpr uint32_t EM = 64 * RT;
    __shared__ __align__(16) uint16_t X[(EM + 4) * EST];
    __shared__ __align__(16) float bias[3 * C];
    __shared__ __align__(16) float sp[EGRP][C];
    __shared__ uint32_t s_len[EM / 2 + 2];
    __shared__ uint16_t s_row[EM / 2 + 2];
    __shared__ uint64_t s_off[EM / 2 + 2];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wc = wave & 1u, wr = wave >> 1;  // this wave's 64 channels and 128 rows
    for (uint32_t i = tid; i < 3 * C; i += 256) {
        const uint32_t l = i / C, c = i % C;
        bias[i] = bf2f(a.theta_b[(l == 0 ? O_B1 : (l == 1 ? O_B2 : O_B3)) + c]);
    }
    // the zero border: two rows before the tile and two after
    for (uint32_t i = tid; i < 4 * EST; i += 256) X[(i < 2 * EST ? 0 : EM * EST) + i] = 0;
    const uint32_t nt = *a.n_tiles;
    for (uint32_t ti = blockIdx.x; ti < nt; ti += gridDim.x) {
        const uint4 t = a.tiles[ti];
        const uint32_t first = t.x, cnt = t.y;  // cnt <= EM / 2 + 1: two rows at least per sequence
        __syncthreads();
        if (tid < cnt) {
            s_len[tid] = min(a.len[first + tid], a.P);
            s_row[tid] = a.rstart[first + tid];
            s_off[tid] = a.off[TRAIN ? a.rows[first + tid] : first + tid];
        }
        __syncthreads();
        if (EM == 256 || tid < EM) {
            // embedding: thread = row
            const uint32_t lo = seq_of_row(s_row, cnt, tid), p = tid - s_row[lo];
            u32x4 e[4] = {};
            if (p < s_len[lo]) {
                const u32x4 *src = (const u32x4 *)(a.theta_b + O_EMB + (uint32_t)a.vocab[a.seq[s_off[lo] + p]] * C0);
#pragma unroll
                for (int k = 0; k < 4; ++k) e[k] = src[k];
            }
            u32x4 *dst = (u32x4 *)(X + (tid + 2) * EST);
#pragma unroll
            for (int k = 0; k < 4; ++k) dst[k] = e[k];
            if (TRAIN) {
                u32x4 *g = (u32x4 *)(a.X0 + (size_t)(t.z + tid) * C0);
                if (tid < t.w)
#pragma unroll
                    for (int k = 0; k < 4; ++k) g[k] = e[k];
                if (tid + EM < t.w)
#pragma unroll
                    for (int k = 0; k < 4; ++k) g[EM * C0 / 8 + k] = u32x4{};
            }
        }
        // validity of this lane's four rows (row wr * 128 + 32 j + lane % 32)
        uint32_t valid = 0;
#pragma unroll
        for (uint32_t j = 0; j < RT; ++j) {
            const uint32_t row = wr * (32 * RT) + 32 * j + (lane & 31u);
            const uint32_t lo = seq_of_row(s_row, cnt, row);
            if (row - s_row[lo] < s_len[lo]) valid |= 1u << j;
        }
        __syncthreads();
        const uint16_t *Xw = X + wr * (32 * RT) * EST;
        const u32x4 *wp = (const u32x4 *)a.pack + wc * 128;
#pragma unroll 1
        for (uint32_t l = 0; l < 3; ++l) {
            f32x16 acc[2][RT];
            if (l == 0) enc_conv<C0, RT>(Xw, wp, lane, acc);
            else enc_conv<C, RT>(Xw, wp + (EKS1 + (l - 1) * EKS) * 256, lane, acc);
            __syncthreads();  // every wave has read the layer's input
            uint2 *h = TRAIN ? a.H[l] + (size_t)ti * (2048 * RT) + wave * (512 * RT) + lane : nullptr;
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t ch = wc * 64 + i * 32 + 8 * q + 4 * (lane >> 5);
                    const float4 b = *(const float4 *)(bias + l * C + ch);
#pragma unroll
                    for (int j = 0; j < RT; ++j) {
                        const float x0 = acc[i][j][4 * q] + b.x, x1 = acc[i][j][4 * q + 1] + b.y,
                                    x2 = acc[i][j][4 * q + 2] + b.z, x3 = acc[i][j][4 * q + 3] + b.w;
                        if (TRAIN)
                            h[((i * RT + j) * 4 + q) * 64] = make_uint2((uint32_t)f2bf(x0) | ((uint32_t)f2bf(x1) << 16),
                                                                       (uint32_t)f2bf(x2) | ((uint32_t)f2bf(x3) << 16));
                        const float g0 = gelu(x0), g1 = gelu(x1), g2 = gelu(x2), g3 = gelu(x3);
                        const bool v = (valid >> j) & 1u;
                        uint2 o;
                        o.x = v ? (uint32_t)f2bf(g0) | ((uint32_t)f2bf(g1) << 16) : 0u;
                        o.y = v ? (uint32_t)f2bf(g2) | ((uint32_t)f2bf(g3) << 16) : 0u;
                        *(uint2 *)(X + (2 + wr * (32 * RT) + 32 * j + (lane & 31u)) * EST + ch) = o;
                    }
                }
            __syncthreads();
            if (TRAIN && l < 2) enc_store_rows(X, (l ? a.A2 : a.A1) + (size_t)t.z * C, t.w, tid);
        }
        // head, EGRP sequences a round: mean over the letters (a wave per
        // sequence, two channels per lane), projection, L2 norm
        for (uint32_t s0 = 0; s0 < cnt; s0 += EGRP) {
#pragma unroll
            for (uint32_t r = 0; r < EGRP / 4; ++r) {
                const uint32_t s = s0 + r * 4 + wave;
                if (s < cnt) {
                    const uint32_t L = s_len[s];
                    const uint16_t *src = X + (2 + s_row[s]) * EST + 2 * lane;
                    float a0 = 0.f, a1 = 0.f;
                    for (uint32_t p = 0; p < L; ++p) {
                        const uint32_t v = *(const uint32_t *)(src + p * EST);
                        a0 += bf2f((uint16_t)v);
                        a1 += bf2f((uint16_t)(v >> 16));
                    }
                    const float inv = L ? 1.f / (float)L : 0.f;
                    a0 *= inv;
                    a1 *= inv;
                    *(float2 *)(&sp[r * 4 + wave][2 * lane]) = make_float2(a0, a1);
                    if (TRAIN) *(float2 *)(a.pool + (size_t)(first + s) * C + 2 * lane) = make_float2(a0, a1);
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            float u[EGRP / 4];
            const float b0 = bf2f(a.theta_b[O_BP + lane]);
#pragma unroll
            for (uint32_t r = 0; r < EGRP / 4; ++r) u[r] = b0;
#pragma unroll 4
            for (uint32_t o = 0; o < C; o += 4) {
                const uint32_t wa = a.wp2[(o / 2) * D + lane], wb = a.wp2[(o / 2 + 1) * D + lane];
#pragma unroll
                for (uint32_t r = 0; r < EGRP / 4; ++r) {
                    const float4 p4 = *(const float4 *)(&sp[r * 4 + wave][o]);
                    u[r] += bf2f((uint16_t)wa) * p4.x;
                    u[r] += bf2f((uint16_t)(wa >> 16)) * p4.y;
                    u[r] += bf2f((uint16_t)wb) * p4.z;
                    u[r] += bf2f((uint16_t)(wb >> 16)) * p4.w;
                }
            }
#pragma unroll
            for (uint32_t r = 0; r < EGRP / 4; ++r) {
                const uint32_t s = s0 + r * 4 + wave;
                float ss = u[r] * u[r];
#pragma unroll
                for (int k = 32; k > 0; k >>= 1) ss += __shfl_xor(ss, k, 64);
                const float nrm = fmaxf(sqrtf(ss), 1e-6f);
                const float zz = u[r] / nrm;
                if (s < cnt) {
                    if (a.z) a.z[(size_t)(first + s) * D + lane] = zz;
                    if (a.zb) a.zb[(size_t)(first + s) * D + lane] = f2bf(zz);
                    if (TRAIN && lane == 0) a.nrm[first + s] = nrm;
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        }
    }
}

// ---------------------------------------------------------------------------
// Training: loss and head, data gradients, weight gradients, their sums.

constexpr uint32_t HP = 16;                        // pairs per round of the head's backward pass
constexpr uint32_t HPART = D * C + D + 4;          // one block's projection gradients and loss
constexpr uint32_t HBLOCKS = 256;                  // most blocks of the head's backward pass
constexpr uint32_t BPART = NTOK * C0 + 3 * C;      // one block's embedding and bias gradients

// Contrastive loss of pair i (sequences 2i, 2i+1; none where the label is below
// zero or no number), back through the norm and the projection to the pooled
// means (dp, already divided by the length), and the projection's gradients.
// A wave takes four pairs of a round of HP; the
// block then adds the round's du x pool into 32 accumulators per thread.
// Latency-bound (4,096 pairs are one round a block); the sums over
// pairs stay in registers and leave as one partial per block, since one atomic
// word per pair (the loss) took 49 us.  With the three kernels it replaces:
// 4,096 pairs 306 -> 24 us.
__global__ __launch_bounds__(256) void k_pair_head(const float *z, const float *nrm, const float *pool,
                                                   const uint32_t *blen, const float *y, uint32_t npairs, float margin,
                                                   float inv_b, const uint32_t *wp2, float *dp, float *part)
{
    __shared__ __align__(16) float sdu[2 * HP][D];
    __shared__ __align__(16) float spool[2 * HP][C];
    __shared__ uint32_t swp[D][C / 2 + 1];  // (output, input pair)
    __shared__ float sloss[4];
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    for (uint32_t i = tid; i < D * C / 2; i += 256) swp[i % D][i / D] = wp2[i];
    float acc[4][8] = {}, accb = 0.f, lsum = 0.f;
    const uint32_t tj = (tid >> 4) * 4, to = (tid & 15u) * 8;
    for (uint32_t p0 = blockIdx.x * HP; p0 < npairs; p0 += gridDim.x * HP) {
        __syncthreads();
        const uint32_t ns = min(2 * HP, 2 * (npairs - p0));  // sequences of this round
        for (uint32_t i = tid; i < 2 * HP * C / 4; i += 256) {
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (i / (C / 4) < ns) v = *(const float4 *)(pool + (size_t)2 * p0 * C + 4 * i);
            *(float4 *)(&spool[0][0] + 4 * i) = v;
        }
#pragma unroll
        for (uint32_t k = 0; k < HP / 4; ++k) {
            const uint32_t q = w * (HP / 4) + k, i = p0 + q;
            float du0 = 0.f, du1 = 0.f;
            if (i < npairs) {
                const float yi = y[i], z0 = z[(size_t)(2 * i) * D + lane], z1 = z[(size_t)(2 * i + 1) * D + lane];
                const float n0 = nrm[2 * i], n1 = nrm[2 * i + 1], diff = z0 - z1;
                float d2 = diff * diff;
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) d2 += __shfl_xor(d2, o, 64);
                float g = 0.f;  // dz0 = g, dz1 = -g
                if (yi >= 0.f) {
                    const float d = sqrtf(d2 + 1e-12f), hinge = fmaxf(0.f, margin - d);
                    lsum += yi * d2 + (1.f - yi) * hinge * hinge;
                    g = (2.f * yi - (1.f - yi) * 2.f * hinge / d) * inv_b * diff;
                }
                float a = z0 * g, b = z1 * g;
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) {
                    a += __shfl_xor(a, o, 64);
                    b += __shfl_xor(b, o, 64);
                }
                du0 = (g - z0 * a) / n0;
                du1 = (z1 * b - g) / n1;
            }
            sdu[2 * q][lane] = du0;
            sdu[2 * q + 1][lane] = du1;
        }
        __syncthreads();
        // dp of this wave's eight sequences, two channels per lane
        {
            float d0[HP / 2] = {}, d1[HP / 2] = {};
#pragma unroll 4
            for (uint32_t j = 0; j < D; j += 4) {
                uint32_t v[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] = swp[j + k][lane];
#pragma unroll
                for (uint32_t s = 0; s < HP / 2; ++s) {
                    const float4 u = *(const float4 *)(&sdu[w * (HP / 2) + s][j]);
                    const float uu[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        d0[s] += bf2f((uint16_t)v[k]) * uu[k];
                        d1[s] += bf2f((uint16_t)(v[k] >> 16)) * uu[k];
                    }
                }
            }
#pragma unroll
            for (uint32_t s = 0; s < HP / 2; ++s) {
                const uint32_t q = w * (HP / 2) + s;
                if (q < ns) {
                    const uint32_t L = blen[2 * p0 + q];
                    const float inv = L ? 1.f / (float)L : 0.f;
                    *(float2 *)(dp + (size_t)(2 * p0 + q) * C + 2 * lane) = make_float2(d0[s] * inv, d1[s] * inv);
                }
            }
        }
#pragma unroll 4
        for (uint32_t s = 0; s < 2 * HP; ++s) {
            const float4 u = *(const float4 *)(&sdu[s][tj]);
            const float4 a = *(const float4 *)(&spool[s][to]), b = *(const float4 *)(&spool[s][to + 4]);
            const float uu[4] = {u.x, u.y, u.z, u.w}, pp[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int o = 0; o < 8; ++o) acc[i][o] += uu[i] * pp[o];
            if (tid < D) accb += sdu[s][tid];
        }
    }
    float *out = part + (size_t)blockIdx.x * HPART;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int o = 0; o < 8; o += 4)
            *(float4 *)(out + (tj + i) * C + to + o) =
                make_float4(acc[i][o], acc[i][o + 1], acc[i][o + 2], acc[i][o + 3]);
    if (tid < D) out[D * C + tid] = accb;
    if (lane == 0) sloss[w] = lsum;
    __syncthreads();
    if (tid < 4) out[D * C + D + tid] = sloss[tid] * inv_b;
}

struct BwdArgs {
    const uint8_t *seq;
    const uint64_t *off;
    const uint32_t *rows, *len;   // row and length of each sequence
    const uint4 *tiles;
    const uint32_t *n_tiles;
    const uint16_t *rstart;
    const uint8_t *vocab;
    const uint16_t *pack;         // transposed weights (k_enc_pack)
    const uint2 *H[3];
    const float *dp;
    uint16_t *dH[3];              // out: pre-activation gradients, packed rows
    float *part;                  // out: BPART sums per block
};

// Packed rows [0, used) of a pre-activation gradient to HBM, and its column
// sums (the bias gradient) into sb.
__device__ __forceinline__ void bwd_store_rows(const uint16_t *X, uint16_t *out, uint32_t used, uint32_t tid, float *sb)
{
    float sum[8] = {};
    for (uint32_t r = tid >> 4; r < used; r += 16) {
        const u32x4 v = *(const u32x4 *)(X + (r + 2) * EST + (tid & 15u) * 8);
        *(u32x4 *)(out + (size_t)r * C + (tid & 15u) * 8) = v;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            sum[2 * k] += bf2f((uint16_t)v[k]);
            sum[2 * k + 1] += bf2f((uint16_t)(v[k] >> 16));
        }
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        sum[k] += __shfl_xor(sum[k], 16, 64);
        sum[k] += __shfl_xor(sum[k], 32, 64);
        if ((tid & 63u) < 16u) atomicAdd(&sb[(tid & 15u) * 8 + k], sum[k]);
    }
}

// Four gradients times the GELU's derivative at four saved pre-activations,
// as bfloat16; zero where the row is no letter.
__device__ __forceinline__ uint2 times_grad(float a, float b, float c, float d, uint2 h, bool v)
{
    const float g0 = a * gelu_grad(bf2f((uint16_t)h.x)), g1 = b * gelu_grad(bf2f((uint16_t)(h.x >> 16))),
                g2 = c * gelu_grad(bf2f((uint16_t)h.y)), g3 = d * gelu_grad(bf2f((uint16_t)(h.y >> 16)));
    return make_uint2(v ? (uint32_t)f2bf(g0) | ((uint32_t)f2bf(g1) << 16) : 0u,
                      v ? (uint32_t)f2bf(g2) | ((uint32_t)f2bf(g3) << 16) : 0u);
}

// Data gradients of a tile, in LDS as in k_encode (same tiles and lane
// mapping): dH3 from dp, then each layer's transposed convolution times the
// GELU's derivative at the saved pre-activation, and the first layer's input
// gradient added per token.  Gradients leave for k_wgrad row by row; bias and
// embedding sums stay in LDS over a block's tiles.
// MFMA-bound like k_encode.  4,096 pairs of protein rows: head's last part,
// three data-gradient products, three bias sums and the embedding scatter
// took 870 us as eight launches over padded rows; 157 us here.
template <int RT>
__global__ __launch_bounds__(256, enc_blocks_per_cu(RT)) void k_enc_bwd(BwdArgs a)
{
    constexpr uint32_t EM = 64 * RT;
    __shared__ __align__(16) uint16_t X[(EM + 4) * EST];
    __shared__ float semb[C0 * (NTOK + 1)];  // [channel][token]
    __shared__ float sbias[3 * C];
    __shared__ uint32_t s_len[EM / 2 + 2], s_seq[EM / 2 + 2];
    __shared__ uint16_t s_row[EM / 2 + 2];
    __shared__ uint8_t s_tok[EM];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wc = wave & 1u, wr = wave >> 1;
    for (uint32_t i = tid; i < C0 * (NTOK + 1); i += 256) semb[i] = 0.f;
    for (uint32_t i = tid; i < 3 * C; i += 256) sbias[i] = 0.f;
    for (uint32_t i = tid; i < 4 * EST; i += 256) X[(i < 2 * EST ? 0 : EM * EST) + i] = 0;
    const uint32_t nt = *a.n_tiles;
    for (uint32_t ti = blockIdx.x; ti < nt; ti += gridDim.x) {
        const uint4 t = a.tiles[ti];
        const uint32_t first = t.x, cnt = t.y;
        __syncthreads();
        if (tid < cnt) {
            s_len[tid] = a.len[first + tid];
            s_row[tid] = a.rstart[first + tid];
            s_seq[tid] = a.rows[first + tid];
        }
        __syncthreads();
        if (EM == 256 || tid < EM) {
            const uint32_t q = seq_of_row(s_row, cnt, tid), p = tid - s_row[q];
            s_tok[tid] = p < s_len[q] ? a.vocab[a.seq[a.off[s_seq[q]] + p]] : (uint8_t)255;
        }
        uint32_t valid = 0;
#pragma unroll
        for (uint32_t j = 0; j < RT; ++j) {
            const uint32_t row = wr * (32 * RT) + 32 * j + (lane & 31u);
            const uint32_t q = seq_of_row(s_row, cnt, row);
            const bool v = row - s_row[q] < s_len[q];
            if (v) valid |= 1u << j;
            const float *dp = a.dp + (size_t)(first + q) * C + wc * 64 + 4 * (lane >> 5);
            const uint2 *h = a.H[2] + (size_t)ti * (2048 * RT) + wave * (512 * RT) + lane;
            uint16_t *x = X + (2 + row) * EST + wc * 64 + 4 * (lane >> 5);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int q2 = 0; q2 < 4; ++q2) {
                    const uint2 hv = h[((i * RT + j) * 4 + q2) * 64];
                    const float4 d = *(const float4 *)(dp + i * 32 + 8 * q2);
                    *(uint2 *)(x + i * 32 + 8 * q2) = times_grad(d.x, d.y, d.z, d.w, hv, v);
                }
        }
        __syncthreads();
        const uint16_t *Xw = X + wr * (32 * RT) * EST;
        const u32x4 *wp = (const u32x4 *)a.pack + wc * 128;
#pragma unroll 1
        for (int l = 1; l >= 0; --l) {
            bwd_store_rows(X, a.dH[l + 1] + (size_t)t.z * C, t.w, tid, sbias + (l + 1) * C);
            f32x16 acc[2][RT];
            enc_conv<C, RT, true>(Xw, wp + (1 - l) * (BLAYER / 8), lane, acc);
            __syncthreads();  // every wave has read the layer's gradient
            const uint2 *h = a.H[l] + (size_t)ti * (2048 * RT) + wave * (512 * RT) + lane;
#pragma unroll
            for (int j = 0; j < RT; ++j) {
                const bool v = (valid >> j) & 1u;
                uint16_t *x = X + (2 + wr * (32 * RT) + 32 * j + (lane & 31u)) * EST + wc * 64 + 4 * (lane >> 5);
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int q2 = 0; q2 < 4; ++q2)
                        *(uint2 *)(x + i * 32 + 8 * q2) =
                            times_grad(acc[i][j][4 * q2], acc[i][j][4 * q2 + 1], acc[i][j][4 * q2 + 2],
                                       acc[i][j][4 * q2 + 3], h[((i * RT + j) * 4 + q2) * 64], v);
            }
            __syncthreads();
        }
        bwd_store_rows(X, a.dH[0] + (size_t)t.z * C, t.w, tid, sbias);
        // input gradient, 32 channels: row tiles wave and wave + 4
        constexpr int NG = (2 * RT + 3) / 4;
        f32x16 g[NG];
#pragma unroll
        for (int j = 0; j < NG; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) g[j][r] = 0.f;
        const uint16_t *xr = X + (wave * 32 + (lane & 31u)) * EST + (lane >> 5) * 8;
        const u32x4 *w1 = (const u32x4 *)a.pack + 2 * (BLAYER / 8);
        u32x4 wq[C / 16];  // a tap's fragments, loaded a tap ahead (past the last: the padding)
#pragma unroll
        for (uint32_t c = 0; c < C / 16; ++c) wq[c] = w1[c * 64 + lane];
#pragma unroll 1
        for (uint32_t tp = 0; tp < T; ++tp)
#pragma unroll
            for (uint32_t c = 0; c < C / 16; ++c) {
                const bf16x8 w = __builtin_bit_cast(bf16x8, wq[c]);
                wq[c] = w1[((tp + 1) * (C / 16) + c) * 64 + lane];
#pragma unroll
                for (int j = 0; j < NG; ++j)
                    if (wave + 4 * j < 2 * RT)
                        g[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            w, *(const bf16x8 *)(xr + (T - 1 - tp + j * 128) * EST + c * 16), g[j], 0, 0, 0);
            }
#pragma unroll
        for (int j = 0; j < NG; ++j) {
            if (wave + 4 * j >= 2 * RT) continue;
            const uint32_t tok = s_tok[(wave + 4 * j) * 32 + (lane & 31u)];
            if (tok != 255u)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    atomicAdd(&semb[(8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * (NTOK + 1) + tok], g[j][r]);
        }
    }
    __syncthreads();
    float *out = a.part + (size_t)blockIdx.x * BPART;
    for (uint32_t i = tid; i < NTOK * C0; i += 256) out[i] = semb[(i % C0) * (NTOK + 1) + i / C0];
    for (uint32_t i = tid; i < 3 * C; i += 256) out[NTOK * C0 + i] = sbias[i];
}

// Weight gradients: dW[o][t][c] = sum over packed rows m of dH[m][o] X[m + t - 2][c]
// (the zero rows between sequences make every window plain row offsets).  A
// block owns 128 outputs x 64 channels x 5 taps of layer 3 or 2, or all of
// layer 1, over one split of the rows: 10 MFMA tiles per wave, so that 7
// fragments from LDS feed 10 products and a row is read 2.25 times.  Operands
// have the rows as their inner dimension: fragments come by transposing LDS
// reads of row-major chunks of 64 rows, a tap being a row offset.  Two groups
// of four waves take the chunks in turn and add their sums at the end, which
// halves the partial sums (k_train_sum adds the splits; atomics on one copy
// of the gradients queue).
// 4,096 pairs of protein rows (139k packed rows), three layers: 1,263 us as
// im2col products over padded rows with transposing LDS stores and atomics,
// 68 us here (753 TFLOP/s).
constexpr uint32_t WROWS = 64, WA = C + 32, WB = 64 + 32;  // rows per chunk; LDS row strides
constexpr uint32_t WPART = 4 * 10 * 16 * 64;               // sums of a block (layer 1: two halves)
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr size_t WLDS = sizeof(uint16_t) * 4 * (WROWS * WA + (WROWS + 4) * WB);  // two groups, two buffers

struct WgradArgs {
    const uint16_t *dH[3], *X[3];
    const uint32_t *total;  // packed rows
    uint32_t ns, ns1;       // splits of the rows for layers 3 and 2, for layer 1
    float *part;            // [4 units x ns, then ns1][WPART]
};

// 32 x 16 fragment of a row-major LDS matrix, transposed: lane l gets column
// c + l % 32, rows r + 8 (l / 32) .. + 7.  A transposing read takes four rows
// of 16 columns per group of 16 lanes.
template <uint32_t ST>
__device__ __forceinline__ bf16x8 tr_frag(const uint16_t *lds, uint32_t r, uint32_t c, uint32_t lane)
{
    typedef __attribute__((address_space(3))) s16x4 lds4;
    const uint16_t *p = lds + (r + (lane >> 5) * 8 + ((lane & 15u) >> 2)) * ST + c + ((lane >> 4) & 1u) * 16 + (lane & 3u) * 4;
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4 *)p);
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4 *)(p + 4 * ST));
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    return __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

__global__ __launch_bounds__(512, 2) void k_wgrad(WgradArgs a)
{
    extern __shared__ __align__(16) uint16_t wl[];
    constexpr uint32_t BUF = WROWS * WA + (WROWS + 4) * WB;
    const uint32_t tid = threadIdx.x & 255u, grp = threadIdx.x >> 8, lane = tid & 63u, w = tid >> 6;
    const bool l1 = blockIdx.x >= 4 * a.ns;
    const uint32_t u = l1 ? 4u : blockIdx.x / a.ns, split = l1 ? blockIdx.x - 4 * a.ns : blockIdx.x % a.ns;
    const uint32_t layer = l1 ? 0u : 2u - (u >> 1), c0 = l1 ? 0u : (u & 1u) * 64, ldx = l1 ? C0 : C;
    const uint32_t xw = l1 ? 4u : 8u;  // 16-byte words of an X row that this block takes
    const uint16_t *dH = a.dH[layer], *Xg = a.X[layer] + c0;
    const uint32_t M = *a.total;
    const uint32_t per = ((M + (l1 ? a.ns1 : a.ns) - 1) / (l1 ? a.ns1 : a.ns) + 2 * WROWS - 1) / (2 * WROWS);  // chunk pairs
    const uint64_t b0 = (uint64_t)split * per * (2 * WROWS);
    const uint32_t m_end = (uint32_t)min((uint64_t)M, b0 + (uint64_t)per * (2 * WROWS));  // rows of this split
    uint16_t *base = wl + grp * 2 * BUF;
    const uint32_t wo = (w >> 1) * 64, wx = l1 ? 0u : (w & 1u) * 32;
    f32x16 acc[2][T];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (uint32_t t = 0; t < T; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][t][r] = 0.f;
    u32x4 ra[4], rb[3];
    const auto fetch = [&](uint32_t it) {
        const uint64_t m0 = b0 + (uint64_t)(2 * it + grp) * WROWS;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const uint64_t m = m0 + (tid >> 4) + 16 * k;
            ra[k] = u32x4{};
            if (m < m_end) ra[k] = *(const u32x4 *)(dH + m * C + (tid & 15u) * 8);
        }
#pragma unroll
        for (uint32_t k = 0; k < 3; ++k) {
            const uint32_t i = tid + 256 * k, r = i / xw;
            const uint64_t m = m0 + r;  // row + 2
            rb[k] = u32x4{};
            if (r < WROWS + 4 && m >= 2 && m - 2 < M) rb[k] = *(const u32x4 *)(Xg + (m - 2) * ldx + (i % xw) * 8);
        }
    };
    const auto stage = [&](uint16_t *buf) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) *(u32x4 *)(buf + ((tid >> 4) + 16 * k) * WA + (tid & 15u) * 8) = ra[k];
#pragma unroll
        for (uint32_t k = 0; k < 3; ++k) {
            const uint32_t i = tid + 256 * k, r = i / xw;
            if (r < WROWS + 4) *(u32x4 *)(buf + WROWS * WA + r * WB + (i % xw) * 8) = rb[k];
        }
    };
    const uint32_t n_it = b0 >= M ? 0u : (uint32_t)((m_end - b0 + 2 * WROWS - 1) / (2 * WROWS));
    if (n_it) {
        fetch(0);
        stage(base);
        if (n_it > 1) fetch(1);
    }
    __syncthreads();
    for (uint32_t it = 0; it < n_it; ++it) {
        if (it + 1 < n_it) stage(base + ((it + 1) & 1u) * BUF);
        if (it + 2 < n_it) fetch(it + 2);
        const uint16_t *A = base + (it & 1u) * BUF, *B = A + WROWS * WA;
#pragma unroll
        for (uint32_t ks = 0; ks < WROWS / 16; ++ks) {
            if (l1 && ((ks ^ w) & 1u)) continue;  // layer 1: two waves share an output tile
            const bf16x8 f0 = tr_frag<WA>(A, ks * 16, wo, lane), f1 = tr_frag<WA>(A, ks * 16, wo + 32, lane);
#pragma unroll
            for (uint32_t t = 0; t < T; ++t) {
                const bf16x8 x = tr_frag<WB>(B, ks * 16 + t, wx, lane);
                acc[0][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f0, x, acc[0][t], 0, 0, 0);
                acc[1][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f1, x, acc[1][t], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    // the second group's sums through LDS, five tiles at a time
    float4 *sx = (float4 *)wl;
    float4 *out = (float4 *)(a.part + (size_t)blockIdx.x * WPART);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        if (grp == 1)
#pragma unroll
            for (uint32_t t = 0; t < T; ++t)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    sx[((w * T + t) * 4 + q) * 64 + lane] =
                        make_float4(acc[i][t][4 * q], acc[i][t][4 * q + 1], acc[i][t][4 * q + 2], acc[i][t][4 * q + 3]);
        __syncthreads();
        if (grp == 0)
#pragma unroll
            for (uint32_t t = 0; t < T; ++t)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 v = sx[((w * T + t) * 4 + q) * 64 + lane];
                    out[((w * 10 + i * T + t) * 4 + q) * 64 + lane] =
                        make_float4(acc[i][t][4 * q] + v.x, acc[i][t][4 * q + 1] + v.y, acc[i][t][4 * q + 2] + v.z,
                                    acc[i][t][4 * q + 3] + v.w);
                }
        __syncthreads();
    }
}

// Sums of the partials into the flat gradient (and the loss): 16 columns of
// four floats by 16 row groups per block.  Bound by reading the partials
// (4,096 protein pairs: 46 MB, 15 us).
struct SumArgs {
    const float *wpart, *hpart, *bpart;
    uint32_t ns, ns1, hblocks, bblocks;
    float *grad, *loss;
};
constexpr uint32_t SUM_W = 4 * WPART / 64, SUM_W1 = WPART / 128, SUM_H = (HPART + 63) / 64, SUM_B = BPART / 64;
static_assert(BPART % 64 == 0 && HPART % 4 == 0 && WPART % 64 == 0, "sum blocks");

__global__ __launch_bounds__(256) void k_train_sum(SumArgs a)
{
    __shared__ float4 sh[16][16];
    const uint32_t col = threadIdx.x & 15u, row = threadIdx.x >> 4;
    uint32_t b = blockIdx.x, kind = 0, n, c4, unit = 0;
    size_t stride;
    const float *src;
    if (b < SUM_W) {
        unit = b / (WPART / 64);
        c4 = (b % (WPART / 64)) * 16 + col;
        src = a.wpart + (size_t)unit * a.ns * WPART;
        n = a.ns;
        stride = WPART;
    } else if ((b -= SUM_W) < SUM_W1) {
        // two waves of a block hold the sums of the same outputs
        kind = 1;
        c4 = b * 16 + col;
        c4 += c4 / 2560u * 2560u;
        src = a.wpart + (size_t)4 * a.ns * WPART;
        n = 2 * a.ns1;
        stride = WPART;
    } else if ((b -= SUM_W1) < SUM_H) {
        kind = 2;
        c4 = b * 16 + col;
        src = a.hpart;
        n = 4 * c4 < HPART ? a.hblocks : 0u;
        stride = HPART;
    } else {
        b -= SUM_H;
        kind = 3;
        c4 = b * 16 + col;
        src = a.bpart;
        n = a.bblocks;
        stride = BPART;
    }
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
    for (uint32_t r = row; r < n; r += 16) {
        const size_t at = kind == 1 ? (r >> 1) * stride + (r & 1u) * (2560u * 4) : r * stride;
        const float4 v = *(const float4 *)(src + at + 4 * (size_t)c4);
        s.x += v.x;
        s.y += v.y;
        s.z += v.z;
        s.w += v.w;
    }
    sh[row][col] = s;
    __syncthreads();
    if (row) return;
    for (uint32_t r = 1; r < 16; ++r) {
        const float4 v = sh[r][col];
        s.x += v.x;
        s.y += v.y;
        s.z += v.z;
        s.w += v.w;
    }
    const float v[4] = {s.x, s.y, s.z, s.w};
    if (kind < 2) {
        // word c4 of a block's sums: wave, tile, quarter, lane
        const uint32_t lane = c4 & 63u, q = (c4 >> 6) & 3u, tile = (c4 >> 8) % 10u, w = (c4 >> 8) / 10u;
        const uint32_t o = (w >> 1) * 64 + (tile / T) * 32 + 8 * q + 4 * (lane >> 5), t = tile % T;
        if (kind == 0) {
            const uint32_t c = (unit & 1u) * 64 + (w & 1u) * 32 + (lane & 31u);
            float *g = a.grad + (unit < 2 ? O_W3 : O_W2) + (size_t)o * (T * C) + t * C + c;
#pragma unroll
            for (int k = 0; k < 4; ++k) g[k * T * C] = v[k];
        } else {
            float *g = a.grad + O_W1 + (size_t)o * (T * C0) + t * C0 + (lane & 31u);
#pragma unroll
            for (int k = 0; k < 4; ++k) g[k * T * C0] = v[k];
        }
    } else if (kind == 2) {
        if (4 * c4 < D * C + D) {
#pragma unroll
            for (int k = 0; k < 4; ++k) a.grad[O_WP + 4 * c4 + k] = v[k];
        } else if (4 * c4 < HPART) {
            *a.loss = (v[0] + v[1]) + (v[2] + v[3]);
        }
    } else {
        const uint32_t at = 4 * c4;
        const uint32_t l = (at - NTOK * C0) / C, dst = at < NTOK * C0 ? O_EMB + at
                                                   : (l == 0 ? O_B1 : (l == 1 ? O_B2 : O_B3)) + (at - NTOK * C0) % C;
#pragma unroll
        for (int k = 0; k < 4; ++k) a.grad[dst + k] = v[k];
    }
}

uint32_t nblocks(uint64_t n, uint32_t bs = 256)
{
    uint64_t b = (n + bs - 1) / bs;
    return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(b, 4096));
}

struct Fail {
    int code;
    std::string msg;
};

void hcheck(hipError_t e, const char *what)
{
    if (e != hipSuccess) throw Fail{e == hipErrorOutOfMemory ? IDB_ERR_OOM : IDB_ERR_HIP,
                                    std::string(what) + ": " + hipGetErrorString(e)};
}

}  // namespace

// Embeddings leave for the host in segments of rows, so that copying one
// overlaps computing the next: at most ENC_SEGS segments per launch group of
// ENC_GROUP rows, ENC_SLOTS of them staged at a time (64 MB pinned at most).
constexpr uint32_t ENC_SEGS = 16, ENC_SLOTS = 4, ENC_GROUP = 1u << 20;
constexpr size_t ENC_STAGE_MAX = 64u << 20;  // most input bytes that are staged (and kept on the device)

// ---------------------------------------------------------------------------
// Encoder state: parameters, optimiser moments, and a workspace sized for the
// largest batch seen so far.
struct idb_encoder {
    int device = 0;
    uint32_t P = IDB_ENC_P;  // positions per row: 32 or 160
    hipStream_t stream = nullptr;
    uint8_t vocab[256];
    float *theta = nullptr, *grad = nullptr, *mom1 = nullptr, *mom2 = nullptr;
    uint16_t *theta_b = nullptr;
    uint32_t adam_step = 0;
    std::string err;
    // workspace of a training step
    uint32_t cap_seq = 0;
    uint32_t *blen = nullptr, *brows = nullptr;
    uint16_t *X0 = nullptr, *A[2] = {nullptr, nullptr}, *dH[3] = {nullptr, nullptr, nullptr};
    uint2 *H[3] = {nullptr, nullptr, nullptr};
    float *pool = nullptr, *z = nullptr, *nrm = nullptr, *dp = nullptr, *y = nullptr;
    float *wpart = nullptr, *hpart = nullptr, *bpart = nullptr;  // partial sums
    uint4 *ttiles = nullptr;
    uint16_t *trstart = nullptr;
    uint8_t *vocab_d = nullptr;
    // inference: weights in the fused kernel's order (packed again when the
    // parameters have changed), and the packing of the current rows
    uint16_t *pack = nullptr;
    uint16_t *bpack = nullptr;
    uint32_t *wp2 = nullptr;
    bool pack_stale = true;
    uint4 *tiles = nullptr;
    uint16_t *rstart = nullptr;
    uint32_t *n_tiles = nullptr;
    uint32_t plan_cap = 0;
    float *zbuf = nullptr;
    uint32_t zbuf_cap = 0;
    // host transfers: the second compute stream and the copy stream of an
    // embedding call, pinned staging (inputs and gradients, then the ring of
    // embedding segments), and the device copy of the inputs
    hipStream_t side = nullptr, copy = nullptr;
    hipEvent_t ev_in = nullptr, ev_enc[ENC_SLOTS] = {}, ev_copy[ENC_SLOTS] = {};
    uint8_t *pin = nullptr, *ring = nullptr, *inbuf = nullptr;
    size_t pin_cap = 0, ring_cap = 0, in_cap = 0;
    uint32_t cus = 1;
    std::vector<void *> fixed, ws;  // parameter and workspace allocations
};

namespace {

template <typename T>
T *dalloc(std::vector<void *> &owner, size_t count)
{
    void *p = nullptr;
    hcheck(hipMalloc(&p, std::max<size_t>(count * sizeof(T), 16)), "hipMalloc");
    owner.push_back(p);
    return (T *)p;
}

void free_workspace(idb_encoder *e)
{
    for (void *p : e->ws) (void)hipFree(p);
    e->ws.clear();
    e->cap_seq = 0;
}

// Workspace of a training step over nseq sequences (an even number).  A
// window's tiles hold at least EM + 2 over P + 2 sequences each but its last.
constexpr uint32_t WSPLITS = 56;  // splits of the rows: 4 x 56 + 28 blocks fill 256 CUs

int train_rt(uint32_t P) { return P + 2 <= 66u ? 2 : 4; }

uint32_t tile_capacity(uint32_t nseq, uint32_t P)
{
    const uint32_t windows = (nseq + EPW - 1) / EPW;
    return std::min(nseq, nseq / ((64u * train_rt(P) + 2) / (P + 2)) + windows);
}

void ensure_workspace(idb_encoder *e, uint32_t nseq)
{
    if (nseq <= e->cap_seq) return;
    free_workspace(e);
    const size_t M = (size_t)nseq * (e->P + 2), nt = tile_capacity(nseq, e->P);
    e->blen = dalloc<uint32_t>(e->ws, nseq);
    e->brows = dalloc<uint32_t>(e->ws, nseq);
    e->X0 = dalloc<uint16_t>(e->ws, M * C0);
    for (int l = 0; l < 2; ++l) e->A[l] = dalloc<uint16_t>(e->ws, M * C);
    for (int l = 0; l < 3; ++l) {
        e->dH[l] = dalloc<uint16_t>(e->ws, M * C);
        e->H[l] = dalloc<uint2>(e->ws, nt * 2048 * train_rt(e->P));
    }
    e->pool = dalloc<float>(e->ws, (size_t)nseq * C);
    e->z = dalloc<float>(e->ws, (size_t)nseq * D);
    e->nrm = dalloc<float>(e->ws, nseq);
    e->dp = dalloc<float>(e->ws, (size_t)nseq * C);
    e->y = dalloc<float>(e->ws, nseq / 2);
    e->ttiles = dalloc<uint4>(e->ws, nt);
    e->trstart = dalloc<uint16_t>(e->ws, nseq);
    e->cap_seq = nseq;
}

// The packed weights of the current parameters, on e->stream.
void ensure_pack(idb_encoder *e)
{
    if (!e->pack) {
        // (fragments are read ahead past a pack's end)
        uint16_t *pack = dalloc<uint16_t>(e->fixed, EPACK + EPAD);
        e->bpack = dalloc<uint16_t>(e->fixed, BPACK + EPAD);
        e->wp2 = dalloc<uint32_t>(e->fixed, C / 2 * D);
        e->n_tiles = dalloc<uint32_t>(e->fixed, 2 * ENC_SEGS);
        hcheck(hipMemsetAsync(pack, 0, (EPACK + EPAD) * sizeof(uint16_t), e->stream), "memset");
        hcheck(hipMemsetAsync(e->bpack, 0, (BPACK + EPAD) * sizeof(uint16_t), e->stream), "memset");
        hcheck(hipFuncSetAttribute((const void *)k_wgrad, hipFuncAttributeMaxDynamicSharedMemorySize, (int)WLDS), "wgrad LDS");
        int dev = 0, cus = 0;
        hcheck(hipGetDevice(&dev), "device");
        hcheck(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev), "device");
        e->cus = (uint32_t)std::max(cus, 1);
        e->pack = pack;
    }
    if (e->pack_stale) {
        hipLaunchKernelGGL(k_enc_pack, dim3(256), dim3(256), 0, e->stream, e->theta_b, e->pack, e->wp2, e->bpack);
        e->pack_stale = false;
    }
}

void enc_args(const idb_encoder *e, EncArgs &a, const uint8_t *seq, const uint64_t *off, const uint32_t *len,
              const uint4 *tiles, const uint16_t *rstart, const uint32_t *n_tiles)
{
    a.seq = seq;
    a.off = off;
    a.len = len;
    a.tiles = tiles;
    a.n_tiles = n_tiles;
    a.rstart = rstart;
    a.vocab = e->vocab_d;
    a.theta_b = e->theta_b;
    a.pack = e->pack;
    a.wp2 = e->wp2;
    a.P = e->P;
}

// The packing of n rows of device data, in segments of `rows` rows (a whole
// number of windows), on e->stream.  All segments are planned ahead: a plan
// between two segments would wait for the first one's blocks to leave the CUs.
void embed_plan(idb_encoder *e, const uint32_t *len, uint32_t n, uint32_t rows)
{
    ensure_pack(e);
    if (n > e->plan_cap) {
        hcheck(hipStreamSynchronize(e->stream), "sync");
        (void)hipFree(e->tiles);
        (void)hipFree(e->rstart);
        e->tiles = nullptr;
        e->rstart = nullptr;
        e->plan_cap = 0;
        hcheck(hipMalloc(&e->tiles, sizeof(uint4) * (size_t)n), "hipMalloc");
        hcheck(hipMalloc(&e->rstart, sizeof(uint16_t) * (size_t)n), "hipMalloc");
        e->plan_cap = n;
    }
    hcheck(hipMemsetAsync(e->n_tiles, 0, 2 * ENC_SEGS * sizeof(uint32_t), e->stream), "memset");
    hipLaunchKernelGGL(k_enc_plan<false>, dim3((n + EPW - 1) / EPW), dim3(256), 0, e->stream, len, n, e->P, 256u,
                       (rows + EPW - 1) / EPW, e->tiles, e->n_tiles, e->rstart, PairSource{});
    hcheck(hipGetLastError(), "plan launch");
}

// Embeddings of planned segment seg (`rows` rows each, n in all) by the fused
// kernel on stream s: float32 (z) and/or bfloat16 (zb), 64 per row.
void embed_segment(idb_encoder *e, const uint8_t *seq, const uint64_t *off, const uint32_t *len, uint32_t n,
                   uint32_t rows, uint32_t seg, float *z, uint16_t *zb, hipStream_t s)
{
    const uint32_t first = seg * rows, m = std::min(rows, n - first);
    EncArgs a{};
    enc_args(e, a, seq, off, len, e->tiles + first, e->rstart, e->n_tiles + 2 * seg);
    a.z = z;
    a.zb = zb;
    hipLaunchKernelGGL((k_encode<false, 4>), dim3(std::min(e->cus * enc_blocks_per_cu(4), m)), dim3(256), 0, s, a);
    hcheck(hipGetLastError(), "encoder launch");
}

// Device copies of host inputs for the encoder entry points.
struct DevData {
    idb_dataset d{};
    std::vector<void *> bufs;
    ~DevData()
    {
        for (void *p : bufs) (void)hipFree(p);
    }
    template <typename T>
    const T *up(const T *h, size_t count, hipStream_t s)
    {
        void *p = nullptr;
        hcheck(hipMalloc(&p, std::max<size_t>(count * sizeof(T), 16)), "hipMalloc");
        bufs.push_back(p);
        if (count) hcheck(hipMemcpyAsync(p, h, count * sizeof(T), hipMemcpyHostToDevice, s), "input copy");
        return (const T *)p;
    }
};

const idb_dataset *device_view(const idb_dataset *d, DevData &dd, hipStream_t s)
{
    if (d->mem == IDB_MEM_DEVICE) return d;
    dd.d = *d;
    dd.d.mem = IDB_MEM_DEVICE;
    dd.d.seq = dd.up(d->seq, d->seq_bytes, s);
    dd.d.off = dd.up(d->off, d->n_rows, s);
    dd.d.len = dd.up(d->len, d->n_rows, s);
    return &dd.d;
}

// Pinned memory of at least `bytes` bytes (false: none to be had, the copies
// then go to the caller's arrays directly).
bool pinned(uint8_t **p, size_t *cap, size_t bytes)
{
    if (*cap >= bytes) return true;
    if (*p) (void)hipHostFree(*p);
    *p = nullptr;
    *cap = 0;
    if (hipHostMalloc((void **)p, bytes, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        *p = nullptr;
        return false;
    }
    *cap = bytes;
    return true;
}

// Host inputs of one call on the device: by one copy from pinned staging into
// a buffer that the encoder keeps (five allocations, frees and copies of
// pageable arrays took 0.2 ms a call), or, past ENC_STAGE_MAX bytes, by
// separate copies into memory of the call.
struct Upload {
    idb_encoder *e;
    DevData dd;
    CopyPool::Job jobs[5];
    const void **out[5];
    uint32_t n = 0;
    explicit Upload(idb_encoder *enc) : e(enc) {}
    template <typename T>
    void add(const T *h, size_t count, const T **dst)
    {
        if (count && !h) throw Fail{IDB_ERR_ARG, "missing input array"};
        jobs[n] = {nullptr, h, count * sizeof(T)};
        out[n++] = (const void **)dst;
    }
    void run()
    {
        if (n == 0) return;
        size_t at[5], total = 0;
        for (uint32_t k = 0; k < n; ++k) {
            at[k] = total;
            total += (jobs[k].bytes + 255) & ~(size_t)255;
        }
        total += 256;
        const bool staged = total <= ENC_STAGE_MAX && pinned(&e->pin, &e->pin_cap, total);
        if (staged && e->in_cap < total) {
            (void)hipFree(e->inbuf);
            e->inbuf = nullptr;
            e->in_cap = 0;
            hcheck(hipMalloc((void **)&e->inbuf, total), "hipMalloc");
            e->in_cap = total;
        }
        for (uint32_t k = 0; k < n; ++k) {
            if (staged) *out[k] = e->inbuf + at[k];
            else *out[k] = dd.up((const uint8_t *)jobs[k].src, jobs[k].bytes, e->stream);
            if (staged) jobs[k].dst = e->pin + at[k];
        }
        if (!staged) return;
        CopyPool::get().run(jobs, n);
        hcheck(hipMemcpyAsync(e->inbuf, e->pin, total, hipMemcpyHostToDevice, e->stream), "input copy");
    }
    void add_rows(const idb_dataset *d, idb_dataset &v)
    {
        v = *d;
        if (d->mem == IDB_MEM_DEVICE) return;
        v.mem = IDB_MEM_DEVICE;
        add(d->seq, d->seq_bytes, &v.seq);
        add(d->off, d->n_rows, &v.off);
        add(d->len, d->n_rows, &v.len);
    }
};

// Streams and events of a call in several segments.
void embed_streams(idb_encoder *e)
{
    if (e->copy) return;
    if (!e->ev_in) hcheck(hipEventCreateWithFlags(&e->ev_in, hipEventDisableTiming), "event");
    for (uint32_t k = 0; k < ENC_SLOTS; ++k) {
        if (!e->ev_enc[k]) hcheck(hipEventCreateWithFlags(&e->ev_enc[k], hipEventDisableTiming), "event");
        if (!e->ev_copy[k]) hcheck(hipEventCreateWithFlags(&e->ev_copy[k], hipEventDisableTiming), "event");
    }
    if (!e->side) hcheck(hipStreamCreateWithFlags(&e->side, hipStreamNonBlocking), "stream");
    hcheck(hipStreamCreateWithFlags(&e->copy, hipStreamNonBlocking), "stream");
}

// Nothing of a call is in flight any more when it returns, also by an error.
struct Drain {
    idb_encoder *e;
    ~Drain()
    {
        (void)hipStreamSynchronize(e->stream);
        if (e->side) (void)hipStreamSynchronize(e->side);
        if (e->copy) (void)hipStreamSynchronize(e->copy);
    }
};

// One training step over pairs [first, first + nb) of the (ordered) pair list:
// the gradient into e->grad, the loss behind it.
float step(idb_encoder *e, const idb_dataset *d, const uint32_t *pairs_d, const float *labels_d, const uint32_t *order_d,
           uint64_t first, uint32_t nb, float margin, float inv_b, bool read_loss)
{
    hipStream_t s = e->stream;
    const uint32_t nseq = 2 * nb, nt = tile_capacity(nseq, e->P);
    const int rt = train_rt(e->P);
    ensure_pack(e);
    if (!e->wpart) {
        e->hpart = dalloc<float>(e->fixed, (size_t)HBLOCKS * HPART);
        e->bpart = dalloc<float>(e->fixed, (size_t)e->cus * enc_blocks_per_cu(rt) * BPART);
        e->wpart = dalloc<float>(e->fixed, (size_t)(4 * WSPLITS + WSPLITS / 2) * WPART);
    }
    hcheck(hipMemsetAsync(e->n_tiles, 0, 2 * sizeof(uint32_t), s), "memset");
    const PairSource ps{pairs_d, order_d, labels_d, first, e->brows, e->blen, e->y};
    hipLaunchKernelGGL(k_enc_plan<true>, dim3((nseq + EPW - 1) / EPW), dim3(256), 0, s, d->len, nseq, e->P, 64u * rt, ~0u, e->ttiles,
                       e->n_tiles, e->trstart, ps);
    EncArgs a{};
    enc_args(e, a, d->seq, d->off, e->blen, e->ttiles, e->trstart, e->n_tiles);
    a.z = e->z;
    a.rows = e->brows;
    for (int l = 0; l < 3; ++l) a.H[l] = e->H[l];
    a.X0 = e->X0;
    a.A1 = e->A[0];
    a.A2 = e->A[1];
    a.pool = e->pool;
    a.nrm = e->nrm;
    const dim3 bb(std::min(e->cus * enc_blocks_per_cu(rt), nt));
    if (rt == 2) hipLaunchKernelGGL((k_encode<true, 2>), bb, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((k_encode<true, 4>), bb, dim3(256), 0, s, a);
    const uint32_t hb = std::min(HBLOCKS, (nb + HP - 1) / HP);
    hipLaunchKernelGGL(k_pair_head, dim3(hb), dim3(256), 0, s, e->z, e->nrm, e->pool, e->blen, e->y, nb, margin, inv_b,
                       e->wp2, e->dp, e->hpart);
    BwdArgs b{d->seq, d->off, e->brows, e->blen, e->ttiles, e->n_tiles, e->trstart, e->vocab_d, e->bpack,
              {e->H[0], e->H[1], e->H[2]}, e->dp, {e->dH[0], e->dH[1], e->dH[2]}, e->bpart};
    if (rt == 2) hipLaunchKernelGGL(k_enc_bwd<2>, bb, dim3(256), 0, s, b);
    else hipLaunchKernelGGL(k_enc_bwd<4>, bb, dim3(256), 0, s, b);
    // splits of at least 512 rows
    const uint32_t ns = (uint32_t)std::max<uint64_t>(2, std::min<uint64_t>(WSPLITS, (uint64_t)nseq * (e->P + 2) / 512));
    const uint32_t ns1 = (ns + 1) / 2;
    const WgradArgs wa{{e->dH[0], e->dH[1], e->dH[2]}, {e->X0, e->A[0], e->A[1]}, e->n_tiles + 1, ns, ns1, e->wpart};
    hipLaunchKernelGGL(k_wgrad, dim3(4 * ns + ns1), dim3(512), WLDS, s, wa);
    const SumArgs sa{e->wpart, e->hpart, e->bpart, ns, ns1, hb, bb.x, e->grad, e->grad + N_PARAMS};
    hipLaunchKernelGGL(k_train_sum, dim3(SUM_W + SUM_W1 + SUM_H + SUM_B), dim3(256), 0, s, sa);
    hcheck(hipGetLastError(), "training step launch");
    float l = 0.f;
    if (read_loss) {
        hcheck(hipMemcpyAsync(&l, e->grad + N_PARAMS, sizeof(float), hipMemcpyDeviceToHost, s), "loss");
        hcheck(hipStreamSynchronize(s), "sync");
    }
    return l;
}

template <class F>
int guard(idb_encoder *e, F &&f)
{
    try {
        if (e) hcheck(hipSetDevice(e->device), "hipSetDevice");
        f();
        return IDB_OK;
    } catch (const Fail &x) {
        if (e) e->err = x.msg;
        return x.code;
    } catch (const std::bad_alloc &) {
        if (e) e->err = "host allocation failed";
        return IDB_ERR_OOM;
    } catch (const std::exception &x) {
        if (e) e->err = x.what();
        return IDB_ERR_HIP;
    }
}

}  // namespace

// Embeddings (bfloat16, 64 per row) of rows [0, n) for the learned pair
// kernel.
hipError_t idb_encoder_embed_rows(idb_encoder *e, const uint8_t *seq, const uint64_t *off, const uint32_t *len,
                                  uint32_t n, uint16_t *zb, hipStream_t s)
{
    const int rc = guard(e, [&] {
        hipStream_t keep = e->stream;
        e->stream = s;
        try {
            if (n) {
                embed_plan(e, len, n, n);
                embed_segment(e, seq, off, len, n, n, 0, nullptr, zb, s);
            }
        } catch (...) {
            e->stream = keep;
            throw;
        }
        e->stream = keep;
    });
    return rc == IDB_OK ? hipSuccess : hipErrorUnknown;
}

const char *idb_encoder_error(const idb_encoder *e) { return e ? e->err.c_str() : "no encoder"; }
uint32_t idb_encoder_positions(const idb_encoder *e) { return e ? e->P : 0u; }
int idb_encoder_device(const idb_encoder *e) { return e ? e->device : -1; }

extern "C" {

uint32_t idb_encoder_param_count(void) { return N_PARAMS; }

int idb_encoder_create(int device, const uint8_t *vocab, uint64_t seed, idb_encoder **out)
{
    return idb_encoder_create_positions(device, vocab, IDB_ENC_P, seed, out);
}

int idb_encoder_create_positions(int device, const uint8_t *vocab, uint32_t positions, uint64_t seed,
                                 idb_encoder **out)
{
    if (!out || !vocab) return IDB_ERR_ARG;
    *out = nullptr;
    if (positions != 32 && positions != 160) return IDB_ERR_UNSUPPORTED;
    auto *e = new (std::nothrow) idb_encoder();
    if (!e) return IDB_ERR_OOM;
    e->device = device;
    e->P = positions;
    std::memcpy(e->vocab, vocab, 256);
    for (int b = 0; b < 256; ++b)
        if (e->vocab[b] >= NTOK) {
            delete e;
            return IDB_ERR_ARG;
        }
    const int rc = guard(e, [&] {
        hcheck(hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking), "stream");
        e->theta = dalloc<float>(e->fixed, N_PARAMS);
        e->grad = dalloc<float>(e->fixed, N_PARAMS + 1);  // and the loss
        e->mom1 = dalloc<float>(e->fixed, N_PARAMS);
        e->mom2 = dalloc<float>(e->fixed, N_PARAMS);
        e->theta_b = dalloc<uint16_t>(e->fixed, N_PARAMS);
        e->vocab_d = dalloc<uint8_t>(e->fixed, 256);
        hcheck(hipMemcpyAsync(e->vocab_d, e->vocab, 256, hipMemcpyHostToDevice, e->stream), "vocab");
        // N(0, 1) embedding, U(+-1/sqrt(fan_in)) weights, zero biases
        std::vector<float> h(N_PARAMS, 0.f);
        std::mt19937_64 rng(seed);
        std::normal_distribution<float> nd(0.f, 1.f);
        for (uint32_t i = O_EMB; i < O_W1; ++i) h[i] = nd(rng);
        auto uni = [&](uint32_t o, uint32_t n, uint32_t fan) {
            std::uniform_real_distribution<float> ud(-1.f / std::sqrt((float)fan), 1.f / std::sqrt((float)fan));
            for (uint32_t i = 0; i < n; ++i) h[o + i] = ud(rng);
        };
        uni(O_W1, C * T * C0, T * C0);
        uni(O_W2, C * T * C, T * C);
        uni(O_W3, C * T * C, T * C);
        uni(O_WP, D * C, C);
        hcheck(hipMemcpyAsync(e->theta, h.data(), sizeof(float) * N_PARAMS, hipMemcpyHostToDevice, e->stream), "init");
        hcheck(hipMemsetAsync(e->mom1, 0, sizeof(float) * N_PARAMS, e->stream), "memset");
        hcheck(hipMemsetAsync(e->mom2, 0, sizeof(float) * N_PARAMS, e->stream), "memset");
        hipLaunchKernelGGL(k_to_bf16, dim3(nblocks(N_PARAMS)), dim3(256), 0, e->stream, e->theta, N_PARAMS, e->theta_b);
        hcheck(hipStreamSynchronize(e->stream), "sync");
    });
    if (rc != IDB_OK) {
        idb_encoder_destroy(e);
        return rc;
    }
    *out = e;
    return IDB_OK;
}

void idb_encoder_destroy(idb_encoder *e)
{
    if (!e) return;
    (void)hipSetDevice(e->device);
    if (e->stream) (void)hipStreamSynchronize(e->stream);
    for (void *p : e->fixed) (void)hipFree(p);
    for (void *p : e->ws) (void)hipFree(p);
    (void)hipFree(e->tiles);
    (void)hipFree(e->rstart);
    (void)hipFree(e->zbuf);
    (void)hipFree(e->inbuf);
    if (e->side) (void)hipStreamSynchronize(e->side);
    if (e->copy) (void)hipStreamSynchronize(e->copy);
    if (e->pin) (void)hipHostFree(e->pin);
    if (e->ring) (void)hipHostFree(e->ring);
    if (e->ev_in) (void)hipEventDestroy(e->ev_in);
    for (uint32_t k = 0; k < ENC_SLOTS; ++k) {
        if (e->ev_enc[k]) (void)hipEventDestroy(e->ev_enc[k]);
        if (e->ev_copy[k]) (void)hipEventDestroy(e->ev_copy[k]);
    }
    if (e->side) (void)hipStreamDestroy(e->side);
    if (e->copy) (void)hipStreamDestroy(e->copy);
    if (e->stream) (void)hipStreamDestroy(e->stream);
    delete e;
}

const char *idb_encoder_last_error(const idb_encoder *e) { return idb_encoder_error(e); }

int idb_encoder_get_params(idb_encoder *e, float *host)
{
    if (!e || !host) return IDB_ERR_ARG;
    return guard(e, [&] {
        hcheck(hipMemcpyAsync(host, e->theta, sizeof(float) * N_PARAMS, hipMemcpyDeviceToHost, e->stream), "copy");
        hcheck(hipStreamSynchronize(e->stream), "sync");
    });
}

int idb_encoder_set_params(idb_encoder *e, const float *host)
{
    if (!e || !host) return IDB_ERR_ARG;
    return guard(e, [&] {
        hcheck(hipMemcpyAsync(e->theta, host, sizeof(float) * N_PARAMS, hipMemcpyHostToDevice, e->stream), "copy");
        hipLaunchKernelGGL(k_to_bf16, dim3(nblocks(N_PARAMS)), dim3(256), 0, e->stream, e->theta, N_PARAMS, e->theta_b);
        e->pack_stale = true;
        hcheck(hipMemsetAsync(e->mom1, 0, sizeof(float) * N_PARAMS, e->stream), "memset");
        hcheck(hipMemsetAsync(e->mom2, 0, sizeof(float) * N_PARAMS, e->stream), "memset");
        e->adam_step = 0;
        hcheck(hipStreamSynchronize(e->stream), "sync");
    });
}

int idb_encoder_embed(idb_encoder *e, const idb_dataset *d, float *z_host)
{
    if (!e || !d || !z_host) return IDB_ERR_ARG;
    return guard(e, [&] {
        const uint32_t n = d->n_rows;
        if (n == 0) return;
        Upload up(e);
        idb_dataset v;
        up.add_rows(d, v);
        const Drain drain{e};
        if (std::min(n, ENC_GROUP) > e->zbuf_cap) {
            (void)hipFree(e->zbuf);
            e->zbuf = nullptr;
            e->zbuf_cap = 0;
            hcheck(hipMalloc(&e->zbuf, sizeof(float) * D * std::min(n, ENC_GROUP)), "hipMalloc");
            e->zbuf_cap = std::min(n, ENC_GROUP);
        }
        up.run();
        // Segments of a whole number of packing windows, 4,096 (1 MB) to 65,536
        // rows; neighbours run on two streams, so that one's last tiles share
        // the chip with the next one's first.
        for (uint32_t g0 = 0; g0 < n; g0 += ENC_GROUP) {
            const uint32_t cnt = std::min(ENC_GROUP, n - g0);
            const uint32_t rows = std::min(ENC_GROUP / ENC_SEGS, std::max(4u * EPW, ((cnt + 7) / 8 + EPW - 1) / EPW * EPW));
            const uint32_t segs = (cnt + rows - 1) / rows;
            const size_t slot = sizeof(float) * D * std::min(rows, cnt);
            const bool staged = slot <= ENC_STAGE_MAX / ENC_SLOTS &&
                                pinned(&e->ring, &e->ring_cap, slot * std::min(segs, ENC_SLOTS));
            embed_plan(e, v.len + g0, cnt, rows);
            if (segs > 1) {
                embed_streams(e);
                hcheck(hipEventRecord(e->ev_in, e->stream), "event");
                hcheck(hipStreamWaitEvent(e->side, e->ev_in, 0), "event");
            }
            // while the GPU computes, the caller's pages of the next segment are
            // made present
            const auto present = [&](uint32_t seg) {
                if (!staged || seg >= segs) return;
                const CopyPool::Job job{z_host + (size_t)(g0 + seg * rows) * D, nullptr,
                                        sizeof(float) * D * std::min(rows, cnt - seg * rows)};
                CopyPool::get().run(&job, 1);
            };
            uint32_t issued = 0;
            for (uint32_t done = 0; done < segs; ++done) {
                for (; issued < segs && issued < done + ENC_SLOTS; ++issued) {
                    const uint32_t first = issued * rows, m = std::min(rows, cnt - first), k = issued % ENC_SLOTS;
                    hipStream_t s = issued & 1u ? e->side : e->stream, cs = segs > 1 ? e->copy : s;
                    embed_segment(e, v.seq, v.off + g0, v.len + g0, cnt, rows, issued, e->zbuf, nullptr, s);
                    if (segs > 1) {
                        hcheck(hipEventRecord(e->ev_enc[k], s), "event");
                        hcheck(hipStreamWaitEvent(cs, e->ev_enc[k], 0), "event");
                    }
                    void *dst = staged ? (void *)(e->ring + k * slot) : (void *)(z_host + (size_t)(g0 + first) * D);
                    hcheck(hipMemcpyAsync(dst, e->zbuf + (size_t)first * D, sizeof(float) * D * m, hipMemcpyDeviceToHost,
                                          cs), "copy");
                    if (segs > 1) hcheck(hipEventRecord(e->ev_copy[k], cs), "event");
                }
                const uint32_t first = done * rows, m = std::min(rows, cnt - first), k = done % ENC_SLOTS;
                if (done == 0) present(0);
                present(done + 1);
                hcheck(segs > 1 ? hipEventSynchronize(e->ev_copy[k]) : hipStreamSynchronize(e->stream), "sync");
                if (!staged) continue;
                const CopyPool::Job job{z_host + (size_t)(g0 + first) * D, e->ring + k * slot, sizeof(float) * D * m};
                CopyPool::get().run(&job, 1);
            }
        }
    });
}

int idb_encoder_loss_grad(idb_encoder *e, const idb_dataset *d, const uint32_t *pairs, const float *labels,
                          uint32_t n_pairs, float margin, float *loss, float *grad_host)
{
    if (!e || !d || !pairs || !labels || !loss || !grad_host || n_pairs == 0) return IDB_ERR_ARG;
    return guard(e, [&] {
        for (uint32_t i = 0; i < 2 * n_pairs; ++i)
            if (pairs[i] >= d->n_rows) throw Fail{IDB_ERR_ARG, "pair row out of range"};
        Upload up(e);
        idb_dataset v;
        const uint32_t *pd = nullptr;
        const float *ld = nullptr;
        up.add_rows(d, v);
        up.add(pairs, 2 * (size_t)n_pairs, &pd);
        up.add(labels, (size_t)n_pairs, &ld);
        const Drain drain{e};
        ensure_workspace(e, 2 * n_pairs);
        up.run();
        (void)step(e, &v, pd, ld, nullptr, 0, n_pairs, margin, 1.f / (float)n_pairs, false);
        const size_t bytes = sizeof(float) * (N_PARAMS + 1);
        const CopyPool::Job present{grad_host, nullptr, bytes - sizeof(float)};
        CopyPool::get().run(&present, 1);  // the caller's pages, while the GPU computes
        if (pinned(&e->ring, &e->ring_cap, bytes)) {
            hcheck(hipMemcpyAsync(e->ring, e->grad, bytes, hipMemcpyDeviceToHost, e->stream), "copy");
            hcheck(hipStreamSynchronize(e->stream), "sync");
            std::memcpy(loss, e->ring + bytes - sizeof(float), sizeof(float));
            const CopyPool::Job job{grad_host, e->ring, bytes - sizeof(float)};
            CopyPool::get().run(&job, 1);
        } else {
            hcheck(hipMemcpyAsync(loss, e->grad + N_PARAMS, sizeof(float), hipMemcpyDeviceToHost, e->stream), "copy");
            hcheck(hipMemcpyAsync(grad_host, e->grad, bytes - sizeof(float), hipMemcpyDeviceToHost, e->stream), "copy");
            hcheck(hipStreamSynchronize(e->stream), "sync");
        }
    });
}

int idb_encoder_train(idb_encoder *e, const idb_dataset *d, const uint32_t *pairs, const float *labels,
                      uint64_t n_pairs, const idb_train_params *tp, idb_train_stats *ts)
{
    if (!e || !d || !pairs || !labels || !tp || n_pairs == 0 || tp->batch_pairs == 0 || n_pairs >= (1ull << 32))
        return IDB_ERR_ARG;
    return guard(e, [&] {
        for (uint64_t i = 0; i < 2 * n_pairs; ++i)
            if (pairs[i] >= d->n_rows) throw Fail{IDB_ERR_ARG, "pair row out of range"};
        DevData dd;
        const idb_dataset *dv = device_view(d, dd, e->stream);
        const uint32_t *pd = dd.up(pairs, 2 * (size_t)n_pairs, e->stream);
        const float *ld = dd.up(labels, n_pairs, e->stream);
        const uint32_t B = tp->batch_pairs;
        ensure_workspace(e, 2 * (uint32_t)std::min<uint64_t>(B, n_pairs));
        std::vector<uint32_t> order(n_pairs);
        std::iota(order.begin(), order.end(), 0u);
        std::mt19937_64 rng(tp->seed);
        uint32_t *od = (uint32_t *)dd.up(order.data(), n_pairs, e->stream);
        hipEvent_t t0, t1;
        hcheck(hipEventCreate(&t0), "event");
        hcheck(hipEventCreate(&t1), "event");
        hcheck(hipEventRecord(t0, e->stream), "event");
        const float b1 = 0.9f, b2 = 0.999f;
        uint32_t steps = 0;
        float first_loss = 0.f, last = 0.f;
        double epoch_sum = 0.0;
        uint32_t epoch_n = 0;
        for (uint32_t ep = 0; ep < tp->epochs; ++ep) {
            std::shuffle(order.begin(), order.end(), rng);
            hcheck(hipMemcpyAsync(od, order.data(), sizeof(uint32_t) * n_pairs, hipMemcpyHostToDevice, e->stream),
                   "order");
            // the host copy of `order` is rewritten next epoch: wait for the upload
            hcheck(hipStreamSynchronize(e->stream), "sync");
            epoch_sum = 0.0;
            epoch_n = 0;
            for (uint64_t first = 0; first < n_pairs; first += B) {
                const uint32_t nb = (uint32_t)std::min<uint64_t>(B, n_pairs - first);
                const bool rd = steps == 0 || (tp->log_every && steps % tp->log_every == 0) ||
                                (first + B >= n_pairs);
                const float l = step(e, dv, pd, ld, od, first, nb, tp->margin, 1.f / (float)nb, rd);
                if (rd) {
                    if (steps == 0) first_loss = l;
                    last = l;
                    epoch_sum += l;
                    ++epoch_n;
                }
                ++e->adam_step;
                const float c1 = 1.f - std::pow(b1, (float)e->adam_step), c2 = 1.f - std::pow(b2, (float)e->adam_step);
                hipLaunchKernelGGL(k_adam, dim3(nblocks(N_PARAMS)), dim3(256), 0, e->stream, e->theta, e->grad, e->mom1,
                                   e->mom2, N_PARAMS, tp->lr, b1, b2, 1e-8f, c1, c2, e->theta_b);
                e->pack_stale = true;
                ++steps;
            }
        }
        hcheck(hipEventRecord(t1, e->stream), "event");
        hcheck(hipStreamSynchronize(e->stream), "sync");
        float ms = 0.f;
        (void)hipEventElapsedTime(&ms, t0, t1);
        (void)hipEventDestroy(t0);
        (void)hipEventDestroy(t1);
        if (ts) {
            ts->steps = steps;
            ts->first_loss = first_loss;
            ts->last_loss = last;
            ts->mean_sampled_loss_last_epoch = epoch_n ? (float)(epoch_sum / epoch_n) : 0.f;
            ts->train_ms = ms;
        }
    });
}

}  // extern "C"
