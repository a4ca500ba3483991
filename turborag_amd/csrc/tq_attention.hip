// tq_attention.hip — fused decode attention over compressed pages (turbo_prod
// and turbo_mse) and the turbo_prod logits entry, gfx950.
//
// The reference runs one workgroup per (query row, kv head) that walks every
// token serially (src/cuda/tq_turbo_prod_kernels.cu:439-571,
// src/cuda/tq_turbo_mse_kernels.cu:302-417): 16 workgroups for a GQA 16/2
// decode step.  Here the token range is split (flash-decoding): each wave
// owns one (split, query row, kv head), keeps the reference's online softmax
// over its tokens in the rotated domain, and writes (m, l, acc[D]) partials;
// a combine kernel merges the splits with the usual log-sum-exp rescaling,
// normalises, applies the inverse WHT and the sign flip, and writes fp16.
// Logits follow the reference's convention <q, k> / sqrt(D) (:426, :531,
// turbo_mse :378).
#include <algorithm>
#include <type_traits>

#include "tq_device.h"

namespace tq {
namespace {

using namespace dev;

constexpr float kInitMax = -1e30f;  // kInitMaxLogit, include/tq_shared_device.cuh:10

// Rotated query pair for lane j: qrot = WHT(q * s) * inv (:472-478).
template <int L>
__device__ __forceinline__ void rotate_query(const uint16_t* q, int h, int j, float inv,
                                             float& q0, float& q1) {
    const uint32_t qq = *reinterpret_cast<const uint32_t*>(q + 2 * j);
    const float sh = (h & 1) ? -1.0f : 1.0f;
    q0 = h2f(qq & 0xffff) * sh;
    q1 = h2f(qq >> 16) * (-sh);
    wht_pair<L>(q0, q1, j);
    q0 *= inv;
    q1 *= inv;
}

struct CellPtrs {
    const uint8_t* base;
    size_t cell;
};

__device__ __forceinline__ CellPtrs cell_of(const uint8_t* pool, const int32_t* slots, int t,
                                            int h, const PageGeom& g) {
    int page, tib;
    split_slot(slots[t], g, page, tib);
    return {pool + (size_t)page * g.page_size, (size_t)(tib * g.H + h)};
}

// Where the generic decode finds a row's tokens.  Slot-mapped rows all attend
// tokens [0, n) of one slot list (a negative slot: no token).
struct SlotTokens {
    const int32_t* slots;
    int n;
    struct Row {
        int kv;
    };
    __device__ Row row(int) const { return {n}; }
    __device__ bool cell(const Row&, int t, const PageGeom& g, int& page, int& tib) const {
        const int s = slots[t];
        if (s < 0) return false;
        split_slot(s, g, page, tib);
        return true;
    }
};
// Paged rows: query row q attends the first min(row_kv_len[q], max_kv_len)
// tokens of sequence row_seq[q]; token t is at position t % B of page
// block_tables[seq * max_blocks + t / B] (a negative page: no token).
// max_kv_len <= max_blocks * B (checked on the host) keeps t / B in the row.
struct PagedTokens {
    const int32_t* block_tables;
    const int32_t* row_seq;
    const int32_t* row_kv_len;
    int max_blocks, max_kv_len;
    struct Row {
        int kv, seq;
    };
    __device__ Row row(int q) const { return {min(row_kv_len[q], max_kv_len), row_seq[q]}; }
    __device__ bool cell(const Row& r, int t, const PageGeom& g, int& page, int& tib) const {
        const int blk = g.bs_shift >= 0 ? t >> g.bs_shift : t / g.block_size;
        page = block_tables[(size_t)r.seq * max_blocks + blk];
        tib = t - blk * g.block_size;
        return page >= 0;
    }
};

// ---------------------------------------------------------------------------
// Split-K partial: one wave per (split, row = q*H + h).
// ws[(split * rows + row) * (D + 2) + ...] = acc[0..D), m, l.
// Any head_dim and page geometry (the matrix-core kernels take D = 64 and 128
// with aligned pages).
// ---------------------------------------------------------------------------
template <int D, bool PROD, class Tok>
__global__ __launch_bounds__(64) void attn_partial_kernel(
    const uint16_t* __restrict__ query, const uint8_t* __restrict__ pool, Tok tok,
    float* __restrict__ ws, PageGeom g, int rows, int tokens_per_split, int num_splits,
    float inv) {
    constexpr int L = D / 2;
    __shared__ float tk[16], tv[16];
    const int lane = threadIdx.x;
    if (lane < 16) {
        tk[lane] = PROD ? kK3[lane & 7] : kV4[lane];
        tv[lane] = kV4[lane];
    }
    __syncthreads();
    const int j = lane % L;
    const int split = blockIdx.x % num_splits;
    const int row = blockIdx.x / num_splits;
    const int h = row % g.H;
    const typename Tok::Row tr = tok.row(row / g.H);

    float q0, q1;
    rotate_query<L>(query + (size_t)row * D, h, j, inv, q0, q1);

    const int t0 = split * tokens_per_split;
    const int t1 = min(tr.kv, t0 + tokens_per_split);
    float m = kInitMax, l = 0.0f, a0 = 0.0f, a1 = 0.0f;
    for (int t = t0; t < t1; ++t) {
        int page, tib;
        if (!tok.cell(tr, t, g, page, tib)) continue;  // no token here (wave-uniform)
        const CellPtrs c{pool + (size_t)page * g.page_size, (size_t)(tib * g.H + h)};
        const uint32_t kb = c.base[g.kc_off + c.cell * g.code_stride + j];
        const float ks = h2f(ld_u16(c.base + g.ks_off + c.cell * g.scale_stride));
        const uint32_t n0 = kb & 0xf, n1 = kb >> 4;
        float logit;
        if (PROD) {
            const float re = h2f(ld_u16(c.base + g.kres_off + c.cell * g.scale_stride));
            float s1 = q0 * tk[n0] + q1 * tk[n1];
            float s2 = ((n0 & 8) ? q0 : -q0) + ((n1 & 8) ? q1 : -q1);
            s1 = sum_lanes<L>(s1);
            s2 = sum_lanes<L>(s2);
            logit = (s1 + s2 * re) * ks * inv;
        } else {
            const float s1 = sum_lanes<L>(q0 * tk[n0] + q1 * tk[n1]);
            logit = s1 * ks * inv;
        }
        const float m_new = fmaxf(m, logit);
        const float a = expf(m - m_new), b = expf(logit - m_new);
        l = l * a + b;
        m = m_new;
        const uint32_t vb = c.base[g.vc_off + c.cell * g.code_stride + j];
        const float vs = h2f(ld_u16(c.base + g.vs_off + c.cell * g.scale_stride));
        a0 = a0 * a + b * (tv[vb & 0xf] * vs);
        a1 = a1 * a + b * (tv[vb >> 4] * vs);
    }
    float* out = ws + ((size_t)split * rows + row) * (D + 2);
    if (lane < L) {
        out[2 * j] = a0;
        out[2 * j + 1] = a1;
    }
    if (lane == 0) {
        out[D] = m;
        out[D + 1] = l;
    }
}

// Merge splits, normalise, inverse WHT, sign flip, fp16 (:560-570).
template <int D>
__global__ __launch_bounds__(64) void attn_combine_kernel(const float* __restrict__ ws,
                                                          uint16_t* __restrict__ output,
                                                          PageGeom g, int rows, int num_splits,
                                                          float inv) {
    constexpr int L = D / 2;
    const int lane = threadIdx.x;
    const int j = lane % L;
    const int row = blockIdx.x;
    const int h = row % g.H;
    float M = kInitMax;
    for (int s = 0; s < num_splits; ++s) M = fmaxf(M, ws[((size_t)s * rows + row) * (D + 2) + D]);
    float lsum = 0.0f, a0 = 0.0f, a1 = 0.0f;
    for (int s = 0; s < num_splits; ++s) {
        const float* p = ws + ((size_t)s * rows + row) * (D + 2);
        const float w = expf(p[D] - M);
        lsum += p[D + 1] * w;
        a0 += p[2 * j] * w;
        a1 += p[2 * j + 1] * w;
    }
    const float inv_l = lsum > 0.0f ? 1.0f / lsum : 1.0f;
    a0 *= inv_l;
    a1 *= inv_l;
    wht_pair<L>(a0, a1, j);
    if (lane >= L) return;
    const float s0 = (h & 1) ? -inv : inv;
    const uint32_t o = (uint32_t)f2h(a0 * s0) | ((uint32_t)f2h(a1 * -s0) << 16);
    *reinterpret_cast<uint32_t*>(output + (size_t)row * D + 2 * j) = o;
}

// ---------------------------------------------------------------------------
// turbo_prod logits (:346-434): one thread per kv token, the rotated query of
// the workgroup's row in LDS.  blockIdx.x = row * tiles + tile.
// ---------------------------------------------------------------------------
template <int D>
__global__ __launch_bounds__(256) void prod_logits_kernel(
    const uint16_t* __restrict__ query, const uint8_t* __restrict__ pool,
    const int32_t* __restrict__ slots, float* __restrict__ logits, PageGeom g, int num_kv_tokens,
    int tiles, float inv) {
    constexpr int L = D / 2;
    __shared__ float qs[D];
    __shared__ float tk[8];
    const int row = blockIdx.x / tiles, tile = blockIdx.x % tiles;
    const int h = row % g.H;
    if (threadIdx.x < 8) tk[threadIdx.x] = kK3[threadIdx.x];
    if (threadIdx.x < 64) {
        const int j = threadIdx.x % L;
        float q0, q1;
        rotate_query<L>(query + (size_t)row * D, h, j, inv, q0, q1);
        if (threadIdx.x < L) {
            qs[2 * j] = q0;
            qs[2 * j + 1] = q1;
        }
    }
    __syncthreads();
    const int t = tile * 256 + threadIdx.x;
    if (t >= num_kv_tokens) return;
    if (slots[t] < 0) {  // unmapped token: excluded, like a -inf logit
        logits[(size_t)row * num_kv_tokens + t] = -INFINITY;
        return;
    }
    const CellPtrs c = cell_of(pool, slots, t, h, g);
    const uint8_t* kc = c.base + g.kc_off + c.cell * g.code_stride;
    const float ks = h2f(ld_u16(c.base + g.ks_off + c.cell * g.scale_stride));
    const float re = h2f(ld_u16(c.base + g.kres_off + c.cell * g.scale_stride));
    float s1 = 0.0f, s2 = 0.0f;
#pragma unroll 4
    for (int b = 0; b < D / 2; ++b) {
        const uint32_t kb = kc[b];
        const uint32_t n0 = kb & 0xf, n1 = kb >> 4;
        const float x0 = qs[2 * b], x1 = qs[2 * b + 1];
        s1 = fmaf(x0, tk[n0 & 7], s1);
        s1 = fmaf(x1, tk[n1 & 7], s1);
        s2 += ((n0 & 8) ? x0 : -x0) + ((n1 & 8) ? x1 : -x1);
    }
    logits[(size_t)row * num_kv_tokens + t] = (s1 * ks + s2 * (ks * re)) * inv;
}

// ===========================================================================
// Matrix-core path: D = 64 and 128, query rows in groups of 8.
//
// Per kv head h and row group (8 query rows; up to four groups in
// unit::attn_unit_split_kernel), a workgroup of 8 waves owns a range of
// tokens; each wave takes 32-token chunks.
//   QK: S^T[token][col] = sum_d K[token][d] * Q^T[d][col] with
//       v_mfma_f32_16x16x32_f16.  A = K, decoded from nibbles to fp16 through
//       256-entry LDS tables indexed by code byte; B = the rotated query split
//       into fp16 hi + lo parts, columns 2r (hi) and 2r+1 (lo) of row r, so a
//       single MFMA column pair recovers ~22-bit query precision.  The K3
//       codebook enters as fp16(aK*K3[c]) with aK = 1.2918981, which makes all
//       four magnitudes fp16-exact to 1.4e-5 relative (V4 with aV = 1.5982153
//       to 9.3e-5); the scale is divided out per token.  turbo_prod's residual
//       sign is a second A matrix (+-1, exact) with its own accumulator.
//   softmax: base-2 online softmax per row over the chunk, in the MFMA output
//       layout (lane (col, g) holds tokens 4g..4g+3 of each 16-token tile).
//   PV: O[col][d] += sum_t P'[col][t] V[t][d] with the same MFMA.  The QK
//       output layout is exactly the A-operand layout over 32 tokens (two
//       tiles), so P' = p * vs needs no data movement; it is split hi/lo in
//       the column pair like q.  B = V, whose contraction index (tokens) must
//       run inside a lane: each lane loads dword i of 8 tokens' V cells and
//       interleaves the nibbles of token pairs into bytes, one table lookup
//       per (token pair, d).
// Each workgroup merges its waves, applies the inverse WHT and sign flip to
// its unnormalised partial (linear, so allowed before the split merge), and
// writes (o[128], m, l) per row; a combine kernel takes the weighted sum.
// ===========================================================================
namespace mfma {
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

constexpr float kAlphaK = 1.2918981f;
constexpr float kAlphaV = 1.5982153f;
// turbo_mse K: the fp16 table of aV*V4 alone is exact only to 9.2e-5, which
// logits of magnitude ~40 (outlier channels shared by q and k) turn into
// ~1e-3 output errors.  A second table holds the fp16 residual
// (aV*c - fp16(aV*c)) * 2^kLoShift per code, multiplied by the same query
// operand in its own accumulator and scaled back by 2^-kLoShift.
constexpr int kLoShift = 10;
constexpr float kLoScale = 1.0f / (float)(1 << kLoShift);
constexpr float kLog2e = 1.4426950408889634f;
constexpr int kRows = 8;     // query rows per workgroup (16 MFMA columns, hi/lo)
// Page schemes of the split kernels.
constexpr int kSchMse = 0, kSchProd = 1;
constexpr int kPartStride = 128 + 4;  // QJL: floats per partial row: o[128], m, l, pad (16-B rows)

// Stores of 2 and 4 output halves (an output row may start at any half).
__device__ __forceinline__ void store_h2(uint16_t* p, uint32_t v) {
    typedef uint32_t word __attribute__((aligned(2)));
    *reinterpret_cast<word*>(p) = v;
}
__device__ __forceinline__ void store_h4(uint16_t* p, uint32_t v0, uint32_t v1) {
    typedef uint32_t pair __attribute__((ext_vector_type(2), aligned(2)));
    *reinterpret_cast<pair*>(p) = (pair){v0, v1};
}
__device__ __forceinline__ uint32_t pack_h2(float a, float b) {
    return __builtin_bit_cast(uint32_t, (half2v){(_Float16)a, (_Float16)b});
}
// (x - fp16(x)) * 2^kLoShift (exact in fp32), rounded to fp16 by pack_h2.
__device__ __forceinline__ float lo_part(float x) {
    return (x - (float)(_Float16)x) * (float)(1 << kLoShift);
}
// One 16x16x32 fp16 MFMA: c += a * b (fp32 accumulate).
__device__ __forceinline__ f32x4 mma(half8 a, half8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ half8 as_h8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_bit_cast(half8, (u32x4){a, b, c, d});
}
// Batched decode over paged sequences: query row r belongs to sequence
// row_seq[r] (the 8 rows of an aligned group share one) and attends its
// first row_kv_len[r] tokens; token t of sequence s is in page
// block_tables[s * max_blocks + t / B].
// A unit: the npos consecutive row groups (new-token positions) of one
// sequence from row group `first` on, computed together.  It has one item
// per kv head; each item is n passes (workgroup-wide chunk steps of kPass
// tokens) over the unit's first kv_end tokens, a pass weighing w work units,
// at work positions [start, start + w*n) of its head's work (every head has
// the same work, split into segments per head).
struct PagedUnit {
    // index: the unit's number; seq_kv: the unit's sequence, or in a row
    // group's copy the group's own longest row
    int32_t first, npos, kv_end, start, n, w, index, seq_kv;
};
struct PagedRows {
    const int32_t* block_tables;
    const int32_t* row_seq;
    const int32_t* row_kv_len;
    int max_blocks;
    // The step's plan: plan[0] units, then a sentinel whose start is the total
    // work plan[1], in plan[2] segments per head; a copy of each row group's
    // unit.  From paged_plan_kernel, or (units null: up to unit::kPlanGroups
    // row groups) computed by every split workgroup for itself, the first one
    // leaving group_unit and plan for the merge.
    const PagedUnit* units;
    PagedUnit* group_unit;
    int32_t* plan;
    // A page-sized region of the workspace that masked tokens' loads address
    // (always valid memory; what they read is not used)
    const uint8_t* spare_page;
    uint32_t inv_segments;  // floor((2^32 - 1) / segments per head)
};
// Workgroup s of G takes the work positions [bound(s), bound(s + 1)) with
// bound(s) = floor(s * total / G) = q*s + floor(r*s / G) (q, r = total div, mod
// G; r*s < G*G stays in 32 bits); a pass belongs to the segment holding its
// first work position.  Divisions by G through inv = floor((2^32 - 1) / G): the
// high half of n * inv is n / G or one less (n < 2^31: n (1 + 1/G) / 2^32 < 1).
// total = G (a pass per segment): bound(s) = s.
struct Segments {
    int q, r, G;
    uint32_t inv;
    __device__ Segments(int total, int g, uint32_t inv_g) : G(g), inv(inv_g) {
        q = total == g ? 1 : div((uint32_t)total);
        r = total - q * g;
    }
    __device__ int div(uint32_t n) const {
        const uint32_t d = __umulhi(n, inv);
        return (int)(d + (n - d * (uint32_t)G >= (uint32_t)G ? 1u : 0u));
    }
    __device__ int bound(int s) const { return q * s + (r ? div((uint32_t)(r * s)) : 0); }
    // The segment holding work position x < total: an estimate within one of
    // floor(((x + 1) G - 1) / total), then corrected.
    __device__ int of(int x, int total) const {
        if (total == G) return x;
        int g = (int)(((float)x + 1.0f) * (float)G / (float)total) - 1;
        g = max(0, min(g, G - 1));
        while (g + 1 < G && bound(g + 1) <= x) ++g;
        while (g > 0 && bound(g) > x) --g;
        return g;
    }
};
// ceil(v / w) for a pass weight w (1, 3 or 4), v >= 0.
__device__ __forceinline__ int passes_of(int v, int w) {
    return w == 4 ? (v + 3) >> 2 : w == 3 ? (v + 2) / 3 : v;
}
// Passes [x0, x1) of an item (start S, n passes of weight w) that begin in
// the work range [b0, b1).
__device__ __forceinline__ void item_passes(int S, int n, int w, int b0, int b1, int& x0,
                                            int& x1) {
    x0 = passes_of(max(b0 - S, 0), w);
    x1 = min(n, passes_of(max(b1 - S, 0), w));
}
// Inclusive sum over the lanes of a wave (DPP row shifts and row broadcasts).
__device__ __forceinline__ int wave_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // row_bcast:15
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // row_bcast:31
    return v;
}

// Workgroup barrier for LDS traffic only: waits for this wave's LDS accesses,
// not for its outstanding global loads (which __syncthreads() would drain).
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
// fp16 hi or lo part of x: lo = fp16(x - fp32(fp16(x))) (the difference is exact).
__device__ __forceinline__ _Float16 hi_lo(float x, bool lo) {
    const _Float16 h = (_Float16)x;
    return lo ? (_Float16)(x - (float)h) : h;
}
// The lo parts of (x0, x1) as an fp16 pair, given their hi parts h (fp16
// pair, low half x0's): fp16(x - hi) with v_fma_mix (x * 1 - hi rounded once;
// the difference is exact in fp32), one instruction per half.
__device__ __forceinline__ uint32_t lo_pair(float x0, float x1, uint32_t h) {
    uint32_t r;
    asm("v_fma_mixlo_f16 %0, %1, 1.0, -%3 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %0, %2, 1.0, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]"
        : "=&v"(r)
        : "v"(x0), "v"(x1), "v"(h));
    return r;
}
constexpr uint16_t f16_bits(float x) { return __builtin_bit_cast(uint16_t, (_Float16)x); }
constexpr uint32_t f16_pair(float a, float b) {
    return (uint32_t)f16_bits(a) | ((uint32_t)f16_bits(b) << 16);
}
// (x - fp16(x)) * 2^kLoShift, exact in fp32 (mfma::lo_part at compile time).
constexpr float lo_part_c(float x) { return (x - (float)(_Float16)x) * (float)(1 << kLoShift); }

// fp16 bits of the codebook values the decode tables hold: aK*K3[j],
// aV*V4[j], the lo parts (x - fp16(x)) * 2^kLoShift of aV*V4[j], and those of
// aK*K3[j] unscaled (fp16 subnormals, whose step is 1e-7 of a level).
struct Fp16Tables {
    uint32_t k3[8], k3lo[8], v4[16], v4lo[16];
};
constexpr Fp16Tables make_fp16_tables() {
    Fp16Tables t{};
    for (int j = 0; j < 8; ++j) {
        t.k3[j] = f16_bits(kAlphaK * dev::kK3[j]);
        t.k3lo[j] = f16_bits(kAlphaK * dev::kK3[j] - (float)(_Float16)(kAlphaK * dev::kK3[j]));
    }
    for (int j = 0; j < 16; ++j) {
        t.v4[j] = f16_bits(kAlphaV * dev::kV4[j]);
        t.v4lo[j] = f16_bits(lo_part_c(kAlphaV * dev::kV4[j]));
    }
    return t;
}
constexpr Fp16Tables kF16 = make_fp16_tables();
// The fp16 pair (t[j], t[j + 1]).
template <int N>
constexpr uint32_t f16_pair_of(const uint32_t (&t)[N], int j) {
    return t[j] | (t[j + 1] << 16);
}
// Selector of entry g < 4 of a 4-entry fp16 table held as two fp16 pairs:
// bytes 2g, 2g + 1, then zeros.
__device__ __forceinline__ uint32_t lut4_sel(int g) {
    return (uint32_t)(2 * g) | ((uint32_t)(2 * g + 1) << 8) | 0x0C0C0000u;
}
// t[4m + g] (in the low half) for the 4-entry slice m of t, g given by sel.
template <int N>
__device__ __forceinline__ uint32_t lut4(const uint32_t (&t)[N], int m, uint32_t sel) {
    return __builtin_amdgcn_perm(f16_pair_of(t, 4 * m + 2), f16_pair_of(t, 4 * m), sel);
}
// Decode tables in the one-address-two-pairs layout: S rows (256 B each,
// 32 copies of the entry in bytes 0..127) at byte 0 and K|V rows at byte
// kOffKV (K copies in bytes 0..127, turbo_prod's V copies in 128..255); entry
// b holds the fp16 pairs of code byte b (low nibble = even d):
//   K: turbo_prod (aK*K3[b & 7], aK*K3[(b >> 4) & 7]); turbo_mse the hi
//      parts fp16(aV*V4[b & 15]), fp16(aV*V4[b >> 4]) (its V lookups read them
//      too);
//   S: turbo_prod the residual signs (nibble bit 3 set: +1.0, else -1.0), or
//      with KLO the lo parts of aK*K3; turbo_mse the lo parts of aV*V4;
//   V (turbo_prod): (aV*V4[b & 15], aV*V4[b >> 4]).
// Wave w of 8 writes rows 32w .. 32w + 31 of each table from registers (no
// memory traffic): with those rows one nibble of every entry is uniform
// across the wave and the other comes from a 4-entry fp16 table by v_perm.
//   S rows, and turbo_mse's K rows: store k < 4 writes row 32w + 8k + lane / 8,
//     copies 4q .. 4q + 3 (q = lane % 8): low nibble 8(k % 2) + lane / 8, high
//     nibble 2w + k / 2;
//   turbo_prod's K | V rows: store k < 8 writes row 32w + 4k + lane / 16, group
//     lane % 16 (K copies, then V copies): low nibble 4(k % 4) + lane / 16, high
//     nibble 2w + k / 4.
template <bool PROD>
struct TableWords {
    static constexpr int kR1Stores = PROD ? 8 : 4;
    uint32_t r0[4], r1[kR1Stores];
};
// The lo parts of aV*V4 as pairs: store k < 4 of wave w holds row
// 32w + 8k + lane / 8 (turbo_mse's S rows; turbo_prod's V lo rows).
__device__ __forceinline__ void lo_table_words(int w, int lane, uint32_t (&r)[4]) {
    const int g8 = lane >> 3;
    const uint32_t sel8 = lut4_sel(g8 & 3);
    const bool hi8 = (g8 & 4) != 0;
    uint32_t llo[2];
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
        llo[hh] = hi8 ? lut4(kF16.v4lo, 2 * hh + 1, sel8) : lut4(kF16.v4lo, 2 * hh, sel8);
#pragma unroll
    for (int k = 0; k < 4; ++k) r[k] = llo[k & 1] | (kF16.v4lo[2 * w + (k >> 1)] << 16);
}
template <bool PROD, bool KLO = false>
__device__ __forceinline__ TableWords<PROD> decode_table_words(int w, int lane) {
    TableWords<PROD> tw;
    uint32_t(&r0)[4] = tw.r0;
    uint32_t(&r1)[TableWords<PROD>::kR1Stores] = tw.r1;
    {
        const int g4 = lane >> 4, g8 = lane >> 3;
        const uint32_t sel4 = lut4_sel(g4), sel8 = lut4_sel(g8 & 3);
        const bool hi8 = (g8 & 4) != 0;
        if constexpr (PROD) {
            if constexpr (KLO) {
                const uint32_t lo = hi8 ? lut4(kF16.k3lo, 1, sel8) : lut4(kF16.k3lo, 0, sel8);
#pragma unroll
                for (int k = 0; k < 4; ++k) r0[k] = lo | (kF16.k3lo[(2 * w + (k >> 1)) & 7] << 16);
            } else {
                const uint32_t sh = (w & 4) ? 0x3C000000u : 0xBC000000u;  // row bit 7 = w bit 2
#pragma unroll
                for (int k = 0; k < 4; ++k) r0[k] = ((k & 1) ? 0x3C00u : 0xBC00u) | sh;  // row bit 3
            }
            const bool vq = (lane & 8) != 0;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const uint32_t vpair =
                    lut4(kF16.v4, k & 3, sel4) | (kF16.v4[2 * w + (k >> 2)] << 16);
                const uint32_t kpair =
                    lut4(kF16.k3, k & 1, sel4) | (kF16.k3[(2 * w + (k >> 2)) & 7] << 16);
                r1[k] = vq ? vpair : kpair;
            }
        } else {
            uint32_t vlo[2];
#pragma unroll
            for (int hh = 0; hh < 2; ++hh)
                vlo[hh] = hi8 ? lut4(kF16.v4, 2 * hh + 1, sel8) : lut4(kF16.v4, 2 * hh, sel8);
            lo_table_words(w, lane, r0);
#pragma unroll
            for (int k = 0; k < 4; ++k) r1[k] = vlo[k & 1] | (kF16.v4[2 * w + (k >> 1)] << 16);
        }
    }
    return tw;
}
// The residual signs of a turbo_prod code dword's 8 nibbles (bit 3 set: +1.0,
// else -1.0) as fp16, in registers.
__device__ __forceinline__ half8 sign_octet(uint32_t wd) {
    const uint32_t he = ((wd << 4) & 0x80808080u) ^ 0xBCBCBCBCu;  // even dims' high bytes
    const uint32_t ho = (wd & 0x80808080u) ^ 0xBCBCBCBCu;         // odd dims'
    return as_h8(__builtin_amdgcn_perm(ho, he, 0x040C000Cu), __builtin_amdgcn_perm(ho, he, 0x050C010Cu),
                 __builtin_amdgcn_perm(ho, he, 0x060C020Cu), __builtin_amdgcn_perm(ho, he, 0x070C030Cu));
}
// The factor of a logit's low products (K's and q's lo parts, x 2^kLoShift) for
// a K scale x: 0 beside an infinite one, whose logit takes its sign from the hi
// products (inf - inf otherwise).
__device__ __forceinline__ float low_factor(float x) {
    return __builtin_isinf(x) ? 0.0f : x * kLoScale;
}
// v of the even (odd) lane of this lane's pair.
__device__ __forceinline__ float pair_even(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xA0, 0xF, 0xF, true));
}
__device__ __forceinline__ float pair_odd(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xF5, 0xF, 0xF, true));
}
// Exponent e with x * 2^-e in [0.5, 1); 0 for a zero or non-finite x.
__device__ __forceinline__ int scale_exp(float x) {
    return __builtin_isfinite(x) ? __builtin_amdgcn_frexp_expf(x) : 0;
}
// V's power of two.  P * vs enters PV as an fp16 hi and lo part; with weights
// of at most 1, products below 2^-14 fell among fp16's subnormals (step 6e-8, hi
// and lo alike: V rows of rms 1e-5 were off by 3 ulps of the output).  So a
// wave's softmax reference lies k below its maximum: weights and their sum are
// 2^k times as large, with k such that the largest vs of the wave's tokens times
// 2^k is in [2^13, 2^14), and products keep ~22 bits down to 2^-28 of it.  `top` is the largest fp16 with the exponent of the largest
// finite vs so far; a chunk that passes it lowers k, and the accumulators are
// rescaled as for a new maximum.  Head_dim 64, and the units over a slot map,
// carry it: 0.1-0.2 us of a call (192 rows x 2 heads x 8,192 tokens, head_dim 128:
// 16.4 -> 16.6; 8 rows x 200 tokens, head_dim 64: 6.3 -> 6.4).  The one-group and paged kernels at head_dim 128 have k = 0.
struct VPower {  // wave-uniform
    uint32_t top = 0x3FFu;  // (exponent field 0: subnormals and zeros)
    float k = 28.0f;        // 28 - exponent field
    // For a chunk whose vs (fp16 bits; 0: no token) are vb, one token in lanes l
    // and l + 32.
    __device__ __forceinline__ void raise(uint32_t vb) {
        vb &= 0x7FFFu;
        // above top and finite
        if (!__any(vb - (top + 1u) < 0x7C00u - (top + 1u))) return;
        uint32_t m = vb < 0x7C00u ? vb : 0u;
        const auto over = [&](auto ctrl) {  // the lane's 16-lane row
            m = max(m, (uint32_t)__builtin_amdgcn_mov_dpp((int)m, decltype(ctrl)::value, 0xF, 0xF, true));
        };
        over(std::integral_constant<int, 0xB1>{});   // quad_perm 1032
        over(std::integral_constant<int, 0x4E>{});   // quad_perm 2301
        over(std::integral_constant<int, 0x141>{});  // row_half_mirror
        over(std::integral_constant<int, 0x140>{});  // row_mirror
        top = max((uint32_t)__builtin_amdgcn_readlane((int)m, 0),
                  (uint32_t)__builtin_amdgcn_readlane((int)m, 16)) | 0x3FFu;
        k = __int_as_float(
            __builtin_amdgcn_readfirstlane(__float_as_int(28.0f - (float)(int)(top >> 10))));
    }
};
template <bool PROD>
__device__ __forceinline__ void store_decode_tables(uint32_t* lut, int kv_words, int w, int lane,
                                                    const TableWords<PROD>& tw) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
        *reinterpret_cast<u32x4*>(&lut[(32 * w + 8 * k + (lane >> 3)) * 64 + 4 * (lane & 7)]) =
            (u32x4){tw.r0[k], tw.r0[k], tw.r0[k], tw.r0[k]};
#pragma unroll
    for (int k = 0; k < TableWords<PROD>::kR1Stores; ++k) {
        const int row = PROD ? 32 * w + 4 * k + (lane >> 4) : 32 * w + 8 * k + (lane >> 3);
        const int q = PROD ? lane & 15 : lane & 7;
        *reinterpret_cast<u32x4*>(&lut[kv_words + row * 64 + 4 * q]) =
            (u32x4){tw.r1[k], tw.r1[k], tw.r1[k], tw.r1[k]};
    }
}
}  // namespace mfma

// ---------------------------------------------------------------------------
// turbo_prod logits on the matrix cores (D = 64, 128; :346-434, 628-648).
//
// Per (token, row): logit = ks (s1 + re s2) / sqrt(D), the reference's
// s1*ks + s2*ks*re, with s1 = sum_d q_d K3[c_d] and s2 = sum_d q_d u3_d
// (u3 = +-1: nibble bit 3).  Both are v_mfma_f32_16x16x32_f16 products
// A (16 tokens x 32 dims) x B (32 dims x 16 columns): column 2r + p holds
// query row r's fp16 hi (p = 0) or lo (p = 1) part, so a column pair sums to
// ~22-bit query precision.  For s1, A is K3[c] split the same way into two
// matrices, fp16(K3[c]) and fp16(K3[c] - fp16(K3[c])), both accumulated into
// one fp32 sum (the four hi/lo cross products: ~2^-22 relative); for s2, A is
// the +-1 matrix (exact).
//
// K3 is odd under c -> 7 - c (K3[7 - c] = -K3[c]), so K3[c] = +-mag[m] with
// mag = K3[4..7], m = (c ^ (c < 4 ? 3 : 0)) & 3 and the sign of bit 2.  The
// fp16 values come from v_perm over a 4-entry register table (low bytes of
// the 4 magnitudes in one dword, high bytes in another), selected by m, then
// the sign bit is xor'ed in; the +-1 matrix is 0x3C00 with the sign bit.
//
// A workgroup of 8 waves takes 128 tokens of one kv head and one group of up
// to 8 query rows; wave w takes tokens 16w .. 16w + 15 (one MFMA tile) and
// rotates query row w.  Lane (i, g) = (lane % 16, lane / 16)
// holds A rows of token i over dims 32g .. 32g + 31 (D = 128): the contraction
// runs over the dims in the order (block kk, lane group g, e) -> dim
// 32g + 8kk + e, so each lane's codes of a tile are one 16-byte load (code
// dword kk = block kk).  The MFMA output lane (n, g) holds tokens 4g .. 4g + 3
// of column n; its token scales come from lanes 16g + m (ks) and
// 16g + 4 + m (re) of its own 16-lane row by DPP row broadcast.
// ---------------------------------------------------------------------------
namespace lgt {
using namespace mfma;
constexpr int kWaves = 8, kTilesW = 1, kTile = 16;  // 4.9 us/layer at 32K; 4 x 2: 5.2, 8 x 2: 5.1
constexpr int kTokens = kWaves * kTilesW * kTile;  // tokens per workgroup
constexpr uint16_t f16b(double x) { return __builtin_bit_cast(uint16_t, (_Float16)x); }
constexpr double f16v(double x) { return (double)(_Float16)x; }
constexpr double kmag(int m) { return (double)dev::kK3[4 + m]; }
constexpr uint16_t mag_hi(int m) { return f16b(kmag(m)); }
constexpr uint16_t mag_lo(int m) { return f16b(kmag(m) - f16v(kmag(m))); }
constexpr uint32_t bytes4(uint16_t a, uint16_t b, uint16_t c, uint16_t d, int hi_byte) {
    const int sh = 8 * hi_byte;
    return ((uint32_t)((a >> sh) & 0xFF)) | ((uint32_t)((b >> sh) & 0xFF) << 8) |
           ((uint32_t)((c >> sh) & 0xFF) << 16) | ((uint32_t)((d >> sh) & 0xFF) << 24);
}
// v_perm tables: byte m of the *L word is the low byte of magnitude m's
// fp16 value, byte m of the *H word its high byte.
constexpr uint32_t kHiL = bytes4(mag_hi(0), mag_hi(1), mag_hi(2), mag_hi(3), 0);
constexpr uint32_t kHiH = bytes4(mag_hi(0), mag_hi(1), mag_hi(2), mag_hi(3), 1);
constexpr uint32_t kLoL = bytes4(mag_lo(0), mag_lo(1), mag_lo(2), mag_lo(3), 0);
constexpr uint32_t kLoH = bytes4(mag_lo(0), mag_lo(1), mag_lo(2), mag_lo(3), 1);

// The three A operands of one code dword W (dims of byte k: low nibble ->
// low half of dword k, high nibble -> high half).
struct AOps {
    half8 hi, lo, u3;
};
__device__ __forceinline__ AOps a_ops(uint32_t W, uint32_t hil, uint32_t hih, uint32_t lol,
                                      uint32_t loh) {
    const uint32_t V = ~W;
    const uint32_t t = (V >> 2) & 0x11111111u;                    // 1 where c < 4
    const uint32_t wm = (W ^ (t | (t << 1))) & 0x33333333u;       // m per nibble
    const uint32_t E = wm & 0x03030303u, O = (wm >> 4) & 0x03030303u;
    const uint32_t xs = (V << 5) & 0x80808080u, ys = (V << 1) & 0x80808080u;  // K3 < 0
    const uint32_t x3 = ((V << 4) & 0x80808080u) | 0x3C3C3C3Cu;   // u3 of low nibbles
    const uint32_t y3 = (V & 0x80808080u) | 0x3C3C3C3Cu;          // of high nibbles
    uint32_t h[4], l[4], u[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t sel =
            __builtin_amdgcn_perm(O, E, (uint32_t)(k | k << 8 | (4 + k) << 16 | (4 + k) << 24)) |
            0x04000400u;
        const uint32_t sk = (uint32_t)(0x0C | k << 8 | 0x0C << 16 | (4 + k) << 24);
        const uint32_t sg = __builtin_amdgcn_perm(ys, xs, sk);
        h[k] = __builtin_amdgcn_perm(hih, hil, sel) ^ sg;
        l[k] = __builtin_amdgcn_perm(loh, lol, sel) ^ sg;
        u[k] = __builtin_amdgcn_perm(y3, x3, sk);
    }
    return {as_h8(h[0], h[1], h[2], h[3]), as_h8(l[0], l[1], l[2], l[3]),
            as_h8(u[0], u[1], u[2], u[3])};
}

template <int N>
__device__ __forceinline__ float row_bcast(float v) {  // lane N of each 16-lane row
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + N, 0xF, 0xF,
                                                      false));
}
template <int N>
__device__ __forceinline__ int row_bcast_i(int v) {
    return __builtin_amdgcn_update_dpp(0, v, 0x150 + N, 0xF, 0xF, false);
}

// VEC: the logits rows are 16-byte aligned and num_kv_tokens % 4 == 0.
// D = 64: two blocks kk instead of four (8 code bytes per lane), and a power of
// two per query row that holds its fp16 parts in range whatever its magnitude
// (the fp32 kernel it replaces there took any).  2 heads x 32,768 tokens at D =
// 64, calls in a row from a graph: 8 rows 4.8 us, 16 rows 6.7, against 11.6 and
// 20.9 for one thread per (token, row).
template <bool VEC, int D>
__global__ __launch_bounds__(64 * kWaves) void prod_logits_mfma_kernel(
    const uint16_t* __restrict__ query, const uint8_t* __restrict__ pool,
    const int32_t* __restrict__ slots, float* __restrict__ logits, PageGeom g, int num_queries,
    int num_kv_tokens, float inv) {
    constexpr int kS = D / 32;           // blocks kk
    constexpr bool QSCALE = D == 64;
    __shared__ uint32_t bq[kS][64][4];  // B operands: [block kk][lane][dword], fp16 pairs
    __shared__ float rsc[kRows];         // QSCALE: the rows' power of two
    // Every kernel argument the loads need, fetched in the first batch of
    // scalar loads (one wait) rather than each before its first use.
    asm volatile("" ::"s"(pool), "s"(slots), "s"(logits), "s"(g.page_size), "s"(g.kc_off),
                 "s"(g.ks_off), "s"(g.kres_off), "s"(g.H), "s"(g.bs_shift));
    const int h = blockIdx.y, rg = blockIdx.z;
    const int nrows = min(kRows, num_queries - rg * kRows);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i = lane & 15, gq = lane >> 4;
    const int jl = lane & (D / 2 - 1);  // this lane's pair of a row
    const int t0 = blockIdx.x * kTokens + w * (kTilesW * kTile);
    // Loads first, in dependency order: the wave's two query rows (raw), the
    // slots of the lane's code token (i) and scale token (4 gq + lane % 4) of
    // each tile, then the codes and the one scale (ks for lane % 8 < 4, else
    // re).  Dropped tokens read the query's first bytes (always valid
    // memory); their addresses are selected, then hidden from the optimiser
    // so each value stays one unconditional load.
    constexpr int kRowsW = kRows / kWaves;  // query rows rotated per wave
    uint32_t qq[kRowsW];
#pragma unroll
    for (int e = 0; e < kRowsW; ++e) {
        const int r = w + kWaves * e;
        qq[e] = r < nrows ? *reinterpret_cast<const uint32_t*>(
                                query + ((size_t)(rg * kRows + r) * g.H + h) * D + 2 * jl)
                          : 0u;
    }
    int slot_c[kTilesW], slot_s[kTilesW];
#pragma unroll
    for (int tt = 0; tt < kTilesW; ++tt) {
        const int tc = t0 + kTile * tt + i, ts = t0 + kTile * tt + 4 * gq + (lane & 3);
        slot_c[tt] = tc < num_kv_tokens ? slots[tc] : -1;
        slot_s[tt] = ts < num_kv_tokens ? slots[ts] : -1;
    }
    const uint64_t dummy = reinterpret_cast<uint64_t>(query);
    const uint64_t soff = (lane & 4) ? g.kres_off : g.ks_off;
    typedef uint32_t codes __attribute__((ext_vector_type(kS)));
    typedef uint32_t codes_a4 __attribute__((ext_vector_type(kS), aligned(4)));
    codes code[kTilesW];
    uint16_t sraw[kTilesW];
#pragma unroll
    for (int tt = 0; tt < kTilesW; ++tt) {
        int page, tib;
        split_slot(slot_c[tt] >= 0 ? slot_c[tt] : 0, g, page, tib);
        // (page sizes are below 4 GiB: checked by the launcher)
        uint64_t ac = slot_c[tt] >= 0
                          ? reinterpret_cast<uint64_t>(pool) +
                                (uint64_t)(uint32_t)page * (uint32_t)g.page_size + g.kc_off +
                                (uint32_t)((tib * g.H + h) * g.code_stride + 4 * kS * gq)
                          : dummy;
        split_slot(slot_s[tt] >= 0 ? slot_s[tt] : 0, g, page, tib);
        uint64_t as = slot_s[tt] >= 0
                          ? reinterpret_cast<uint64_t>(pool) +
                                (uint64_t)(uint32_t)page * (uint32_t)g.page_size + soff +
                                (uint32_t)((tib * g.H + h) * g.scale_stride)
                          : dummy;
        asm volatile("" : "+v"(ac), "+v"(as));
        // 4 kS code bytes at a 4-byte aligned address (one multi-dword load;
        // global loads need dword alignment only).
        code[tt] = *reinterpret_cast<const __attribute__((address_space(1))) codes_a4*>(ac);
        sraw[tt] = *reinterpret_cast<const __attribute__((address_space(1))) uint16_t*>(as);
    }

    // Rotate the wave's query rows w + 8e / kWaves (sign flip, orthonormal
    // WHT) while the codes load; lane j holds dims 2j, 2j + 1: block kk = (j / 4) % kS, lane group
    // g = j / (4 kS), dword j % 4 of columns 2r (hi) and 2r + 1 (lo).
    {
        const float sh = (h & 1) ? -1.0f : 1.0f;
        const int kk = (jl >> 2) & (kS - 1), cg = 16 * (jl / (4 * kS));
#pragma unroll
        for (int e = 0; e < kRowsW; ++e) {
            float q0 = h2f(qq[e] & 0xffff) * sh, q1 = h2f(qq[e] >> 16) * (-sh);
            wht_pair<D / 2>(q0, q1, lane);
            q0 *= inv;
            q1 *= inv;
            if constexpr (QSCALE) {
                const int ex = scale_exp(max_lanes<D / 2>(fmaxf(fabsf(q0), fabsf(q1))));
                q0 = __builtin_amdgcn_ldexpf(q0, -ex);
                q1 = __builtin_amdgcn_ldexpf(q1, -ex);
                if (lane == 0) rsc[w + kWaves * e] = __builtin_amdgcn_ldexpf(1.0f, ex);
            }
            const uint32_t hi = pack_h2(q0, q1);
            const int col = 2 * (w + kWaves * e) + cg;
            bq[kk][col][jl & 3] = hi;
            bq[kk][col + 1][jl & 3] = lo_pair(q0, q1, hi);
        }
    }
    // Register tables for the K operands (values in VGPRs: v_perm reads at
    // most one scalar operand).
    uint32_t hil = kHiL, hih = kHiH, lol = kLoL, loh = kLoH;
    asm volatile("" : "+v"(hil), "+v"(hih), "+v"(lol), "+v"(loh));
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
    half8 b[kS];
#pragma unroll
    for (int kk = 0; kk < kS; ++kk)
        b[kk] = __builtin_bit_cast(half8, *reinterpret_cast<const u32x4*>(bq[kk][lane]));

    const int r = i >> 1;
    const float qinv = QSCALE ? inv * rsc[r] : inv;
    const bool writer = (i & 1) == 0 && r < nrows;
    float* const row_out = logits + ((size_t)(rg * kRows + r) * g.H + h) * num_kv_tokens;
#pragma unroll
    for (int tt = 0; tt < kTilesW; ++tt) {
        f32x4 s1 = {0.f, 0.f, 0.f, 0.f}, s2 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < kS; ++kk) {
            const AOps a = a_ops(code[tt][kk], hil, hih, lol, loh);
            s1 = mma(a.hi, b[kk], s1);
            s2 = mma(a.u3, b[kk], s2);
            s1 = mma(a.lo, b[kk], s1);
        }
        // Lane (n, gq): tokens 4 gq + m of column n; rows r = n / 2 summed
        // over the hi/lo column pair, then scaled by the token's ks.
        const float sv = h2f(sraw[tt]);
        const float ksm[4] = {row_bcast<0>(sv), row_bcast<1>(sv), row_bcast<2>(sv),
                              row_bcast<3>(sv)};
        const float rem[4] = {row_bcast<4>(sv), row_bcast<5>(sv), row_bcast<6>(sv),
                              row_bcast<7>(sv)};
        const int okm[4] = {row_bcast_i<0>(slot_s[tt]), row_bcast_i<1>(slot_s[tt]),
                            row_bcast_i<2>(slot_s[tt]), row_bcast_i<3>(slot_s[tt])};
        float out[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            float x = s1[m] + rem[m] * s2[m];
            x += lane_xor<1>(x);
            out[m] = okm[m] < 0 ? -INFINITY : x * ksm[m] * qinv;
        }
        const int tf = t0 + kTile * tt + 4 * gq;
        if (writer) {
            float* dst = row_out + tf;
            if (VEC && tf + 3 < num_kv_tokens) {
                *reinterpret_cast<float4*>(dst) = make_float4(out[0], out[1], out[2], out[3]);
            } else {
#pragma unroll
                for (int m = 0; m < 4; ++m)
                    if (tf + m < num_kv_tokens) dst[m] = out[m];
            }
        }
    }
}
}  // namespace lgt

// ---------------------------------------------------------------------------
// Decode over the reference's unexported QJL-1b pages (src/cuda/
// tq_qjl_kernels.cu), D = 128: 8 waves of 32-token chunks per (split, kv head,
// row group) workgroup; the 16 MFMA columns are the group's 8 query rows as
// fp16 hi and lo parts (columns 2r, 2r + 1), summed after each product.  The A
// operand of QK is the +-1 sign matrix, read as fp16 octets from an LDS table
// indexed by sign byte; the logit is ks * <qrot, signs> (no 1/sqrt(D) beyond
// the rotation's, :254); the rotation's sign flip has no head term.
// ---------------------------------------------------------------------------
namespace qjl {
using namespace mfma;
constexpr int kWaves = 8, kChunk = 32, kPass = kWaves * kChunk;

__global__ __launch_bounds__(64 * kWaves) void attn_qjl_split_kernel(
    const uint16_t* __restrict__ query, const uint8_t* __restrict__ pool,
    const int32_t* __restrict__ slots, float* __restrict__ ws, float inv, int num_queries,
    int num_kv_tokens, int tokens_per_split, int num_splits, PageGeom g) {
    // One region of 256-byte rows per code byte: in bytes 0..127 of row e the 8
    // copies of the fp16 sign octet of sign byte e, in 128..255 the 32 copies of
    // V's fp16 pair aV*V4 (low nibble = even d); lane l reads copy l % 8 or
    // l % 32.  After the token loop the space holds the waves' results.
    __shared__ __attribute__((aligned(256))) uint32_t lut[256 * 64];
    __shared__ float qs[kRows][128];  // the rotated queries
    __shared__ uint4 bqs[4][64];      // QK B operand (fp16 hi/lo q) of k-step s for lane l
    __shared__ uint64_t tko[kWaves][kChunk], tvo[kWaves][kChunk];
    __shared__ float4 tsc[kWaves][kChunk];  // per token: (unused), K scale, vs, bias
    __shared__ float mm[kWaves][kRows], ml[kWaves][kRows];
    __shared__ uint32_t vstage[256];  // the staged V entries
    static_assert(sizeof(float) * kWaves * kRows * 128 <= sizeof(lut), "merge space");
    float(*mo)[kRows][128] = reinterpret_cast<float(*)[kRows][128]>(&lut[0]);

    // Grid (split, kv head, row group), or one dimension of splits x heads when
    // there are more row groups than a grid dimension holds (the first form
    // needs no divisions before the first loads).
    int split, h, rg;
    if (gridDim.x == (unsigned)num_splits) {
        split = blockIdx.x;
        h = blockIdx.y;
        rg = blockIdx.z;
    } else {
        split = blockIdx.x % num_splits;
        const int hr = blockIdx.x / num_splits;
        h = hr % g.H;
        rg = hr / g.H;
    }
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform (scalar)
    const int i = lane & 15, gq = lane >> 4;
    const int t_begin = split * tokens_per_split;
    const int t_end = min(num_kv_tokens, t_begin + tokens_per_split);
    const size_t pid = ((size_t)rg * g.H + h) * num_splits + split;
    // This wave's query row, loaded before anything waits.
    const int qi = min(rg * kRows + w, num_queries - 1);
    const uint32_t qraw =
        *reinterpret_cast<const uint32_t*>(query + ((size_t)qi * g.H + h) * 128 + 2 * lane);

    // A chunk's codes and per-token scales, loaded ahead of its compute.
    struct Chunk {
        uint32_t kw[2];  // K: tile tau, token 16*tau + i, sign bytes 4gq .. 4gq + 3 (k-steps 0 .. 3)
        uint32_t vw[8];  // V: k-index 8gq + e (token below), dword i
        uint16_t ks, vs;  // this lane's token's fp16 scales (raw: still in flight)
        bool valid;
    };
    // Slot of this lane's token in the chunk at t0 (lanes past the range re-read
    // the last token of the range).
    auto load_slot = [&](int t0) -> int {
        return slots[max(min(t0 + (lane & (kChunk - 1)), t_end - 1), 0)];
    };
    // slot -> cell offsets (exchanged through LDS) -> scale and code loads,
    // issued for every lane.  Tokens past the range or with a negative slot read
    // the first bytes of the query instead (always valid memory: the offset of
    // the query from the pool) and get bias -inf.  The loads stay in flight
    // until the chunk is computed.  Each pool byte is read once per row group:
    // non-temporal loads keep the L2 for the slots and queries.
    const uint64_t dummy_off =
        (uint64_t)(reinterpret_cast<uintptr_t>(query) - reinterpret_cast<uintptr_t>(pool));
    auto fetch = [&](int t0, int slot, Chunk& c) {
        c.valid = t0 + (lane & (kChunk - 1)) < t_end && slot >= 0;
        int page, tib;
        split_slot(c.valid ? slot : 0, g, page, tib);
        const uint64_t cell = (uint64_t)(tib * g.H + h);
        const uint64_t pb = (uint64_t)page * g.page_size;
        // Byte offsets from pool (integer selects: no branches around loads).
        const uint64_t so = pb + cell * g.scale_stride;
        c.ks = ld_u16_nt(pool + (c.valid ? so + g.ks_off : dummy_off));
        c.vs = ld_u16_nt(pool + (c.valid ? so + g.vs_off : dummy_off + 2));
        // (lanes l and l + 32 hold the same token; K rows are 16 sign bytes)
        tko[w][lane & (kChunk - 1)] = c.valid ? pb + g.kc_off + cell * 16u : dummy_off;
        tvo[w][lane & (kChunk - 1)] = c.valid ? pb + g.vc_off + cell * g.code_stride : dummy_off;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int tau = 0; tau < 2; ++tau)
            c.kw[tau] = ld_u32_nt(pool + (tko[w][16 * tau + i] + 4 * gq));
        // (the K words first: the QK waits for them while the V words may still
        // be in flight)
        __builtin_amdgcn_sched_barrier(0);
        // k-index 8gq + e is token 4gq + e (e < 4) or 16 + 4gq + (e - 4).
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int tok = e < 4 ? 4 * gq + e : 16 + 4 * gq + (e - 4);
            c.vw[e] = ld_u32_nt(pool + (tvo[w][tok] + 4 * i));
        }
    };

    // Issue order matters (the vector-memory counter is in order): the query row
    // (above), then the first chunk's slots; the tables are built while they are
    // in flight.
    int t0 = t_begin + w * kChunk;
    const int slot0 = load_slot(t0);
    if (w < 4)  // V's entries staged one per thread, replicated after the first barrier
        vstage[tid] = pack_h2(kAlphaV * pick(kV4, tid & 15), kAlphaV * pick(kV4, tid >> 4));
    float q0 = h2f(qraw & 0xffff), q1 = -h2f(qraw >> 16);
    Chunk cur;
    fetch(t0, slot0, cur);  // in flight during the setup below (empty waves: all invalid)
    {  // this wave's rotated query row: qrot = WHT(q * s) * inv
        wht_pair<64>(q0, q1, lane);
        const bool live = rg * kRows + w < num_queries;
        qs[w][2 * lane] = live ? q0 * inv : 0.0f;
        qs[w][2 * lane + 1] = live ? q1 * inv : 0.0f;
    }
    lds_barrier();  // staged entries and rotated queries visible
    // Every wave writes its rows of both tables with conflict-free 1 KB stores.
#pragma unroll
    for (int k = 0; k < 256 / kWaves; k += 4) {
        const int e = w * (256 / kWaves) + k + (lane >> 4);
        uint4 v4;
        if (lane & 8) {
            const uint32_t v = vstage[e];
            v4 = make_uint4(v, v, v, v);
        } else {
            uint32_t wd[4];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                wd[q] = ((e >> (2 * q)) & 1 ? 0x3C00u : 0xBC00u) |
                        ((e >> (2 * q + 1)) & 1 ? 0x3C000000u : 0xBC000000u);
            v4 = make_uint4(wd[0], wd[1], wd[2], wd[3]);
        }
        *reinterpret_cast<uint4*>(&lut[64 * e + 4 * (lane & 15)]) = v4;
    }
    // B operand of QK: column i = row i/2, hi (i even) or lo (i odd) part; k-index
    // 8*gq + e of step s is d = 32*gq + 8*s + e.
    const bool lo_col = (i & 1) != 0;
    if (w < 4) {
        half8 b;
#pragma unroll
        for (int e = 0; e < 8; ++e) b[e] = hi_lo(qs[i >> 1][32 * gq + 8 * w + e], lo_col);
        bqs[w][lane] = __builtin_bit_cast(uint4, b);
    }
    lds_barrier();
    half8 bq[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) bq[s] = __builtin_bit_cast(half8, bqs[s][lane]);
    // A lookup puts the code byte into byte 1 of its table's address (entry
    // stride 256 B) with one v_perm; byte 1 of the base is re-added.
    const uint32_t lutv = (uint32_t)reinterpret_cast<uintptr_t>((lds_u32*)&lut[32 + (lane & 31)]);
    const uint32_t lutq = (uint32_t)reinterpret_cast<uintptr_t>((lds_u32*)&lut[4 * (lane & 7)]);
    auto at = [](uint32_t word, int b, uint32_t base) -> uint32_t {
        return __builtin_amdgcn_perm(word, base, 0x03020000u | ((4u + b) << 8)) + (base & 0xFF00u);
    };
    typedef __attribute__((address_space(3))) u32x4 lds_u32x4;

    float m_run = kInitMax, l_run = 0.0f;
    f32x4 acc[8];
#pragma unroll
    for (int v = 0; v < 8; ++v) acc[v] = (f32x4){0.f, 0.f, 0.f, 0.f};
    bool first = true;
    int slot_nx = load_slot(t0 + kPass);
    while (t0 < t_end) {  // wave-uniform
        {
            const float ks = h2f(cur.ks), vs = h2f(cur.vs);
            tsc[w][lane & (kChunk - 1)] = cur.valid ? make_float4(0.0f, ks * kLog2e, vs, 0.0f)
                                                    : make_float4(0.f, 0.f, 0.f, -INFINITY);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        Chunk nxt;
        const int t1 = t0 + kPass;
        if (t1 < t_end) {  // codes of the next chunk, slots of the one after
            fetch(t1, slot_nx, nxt);
            slot_nx = load_slot(t1 + kPass);
        }
        // The scale rows of this lane's tokens, read before any lookup (LDS reads
        // complete in order: a read issued after the V lookups would wait for
        // all of them).
        float4 scv[2][4];
#pragma unroll
        for (int tau = 0; tau < 2; ++tau)
#pragma unroll
            for (int e = 0; e < 4; ++e) scv[tau][e] = tsc[w][16 * tau + 4 * gq + e];
        // QK: every lookup of the chunk's sign octets before the first MFMA.
        half8 ka[2][4];
#pragma unroll
        for (int tau = 0; tau < 2; ++tau)
#pragma unroll
            for (int s = 0; s < 4; ++s)
                ka[tau][s] = __builtin_bit_cast(
                    half8, *reinterpret_cast<const lds_u32x4*>(at(cur.kw[tau], s, lutq)));
        __builtin_amdgcn_sched_barrier(0);
        f32x4 cs[2];
#pragma unroll
        for (int tau = 0; tau < 2; ++tau) {
            cs[tau] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 4; ++s) cs[tau] = mma(ka[tau][s], bq[s], cs[tau]);
        }
        // The V lookups (B operands of PV) go out now: the softmax below runs
        // while they are in flight.
        uint32_t bv[8][4];  // [N-tile v = d - 8i][token pair]
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t we = cur.vw[2 * q], wo = cur.vw[2 * q + 1];
            const uint32_t lob = (we & 0x0F0F0F0Fu) | ((wo & 0x0F0F0F0Fu) << 4);
            const uint32_t hib = ((we >> 4) & 0x0F0F0F0Fu) | (wo & 0xF0F0F0F0u);
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                bv[2 * b][q] = *reinterpret_cast<const lds_u32*>(at(lob, b, lutv));
                bv[2 * b + 1][q] = *reinterpret_cast<const lds_u32*>(at(hib, b, lutv));
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // Logits (base 2) of tokens 16*tau + 4*gq + e; hi + lo columns summed.
        float lg[2][4];
        float mloc = -INFINITY;
#pragma unroll
        for (int tau = 0; tau < 2; ++tau)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float4 sc = scv[tau][e];
                lg[tau][e] = fmaf(cs[tau][e] + quad_xor<1>(cs[tau][e]), sc.y, sc.w);
                mloc = fmaxf(mloc, lg[tau][e]);
            }
        mloc = lane_xor_reduce<16>(mloc, [](float x, float y) { return fmaxf(x, y); });
        mloc = lane_xor_reduce<32>(mloc, [](float x, float y) { return fmaxf(x, y); });
        // v_exp_f32 without denormal handling: arguments are <= 0 and a weight
        // below 2^-126 of the running maximum is negligible.
        const float m_new = fmaxf(m_run, mloc);
        const float alpha = first ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);
        m_run = m_new;
        float lsum = 0.0f;
#pragma unroll
        for (int tau = 0; tau < 2; ++tau)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                lg[tau][e] = __builtin_amdgcn_exp2f(lg[tau][e] - m_new);
                lsum += lg[tau][e];
            }
        l_run = l_run * alpha + lsum;
        if (!first && __any(alpha != 1.0f)) {
            // acc lane (d, gq) holds columns 4gq..4gq+3 = rows 2gq, 2gq+1.
            const float a0 = __shfl(alpha, 4 * gq), a1 = __shfl(alpha, 4 * gq + 2);
#pragma unroll
            for (int v = 0; v < 8; ++v) {
                acc[v][0] *= a0;
                acc[v][1] *= a0;
                acc[v][2] *= a1;
                acc[v][3] *= a1;
            }
        }
        half8 ap;
#pragma unroll
        for (int e = 0; e < 8; ++e) ap[e] = hi_lo(lg[e >> 2][e & 3] * scv[e >> 2][e & 3].z, lo_col);
#pragma unroll
        for (int v = 0; v < 8; ++v)
            acc[v] = mma(ap, as_h8(bv[v][0], bv[v][1], bv[v][2], bv[v][3]), acc[v]);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        cur = nxt;
        t0 = t1;
        first = false;
    }

    // Wave results: l summed over the g lanes of each column; o rows from the hi
    // + lo columns, the V codebook scale divided out.  Then the waves are merged
    // per row, the inverse WHT and sign flip applied, and the partial written.
    {
        float l_tot = lane_xor_reduce<16>(l_run, [](float x, float y) { return x + y; });
        l_tot = lane_xor_reduce<32>(l_tot, [](float x, float y) { return x + y; });
        if (gq == 0 && !lo_col) {
            mm[w][i >> 1] = m_run;
            ml[w][i >> 1] = l_tot;
        }
    }
    const float iav = 1.0f / kAlphaV;
    __syncthreads();  // every wave is done with the tables mo overwrites
#pragma unroll
    for (int v = 0; v < 8; ++v) {
        mo[w][2 * gq][8 * i + v] = (acc[v][0] + acc[v][1]) * iav;
        mo[w][2 * gq + 1][8 * i + v] = (acc[v][2] + acc[v][3]) * iav;
    }
    __syncthreads();
    const int r = w;  // this wave's row of the group
    float M = mm[0][r];
#pragma unroll
    for (int u = 1; u < kWaves; ++u) M = fmaxf(M, mm[u][r]);
    float L = 0.f, o0 = 0.f, o1 = 0.f;
#pragma unroll
    for (int u = 0; u < kWaves; ++u) {
        const float wt = __builtin_amdgcn_exp2f(mm[u][r] - M);  // (argument <= 0)
        L += ml[u][r] * wt;
        o0 += mo[u][r][2 * lane] * wt;
        o1 += mo[u][r][2 * lane + 1] * wt;
    }
    wht_pair<64>(o0, o1, lane);
    float* part = ws + (pid * kRows + r) * kPartStride;
    part[2 * lane] = o0 * inv;
    part[2 * lane + 1] = o1 * -inv;
    if (lane == 0) {
        part[128] = M;
        part[129] = L;
    }
}
}  // namespace qjl

// ---------------------------------------------------------------------------
// Decode of units of up to four row groups (kNP positions of 8 query rows)
// that share every decoded K/V chunk: the new tokens of one paged sequence
// (PAGED), or consecutive row groups over one slot map (many query rows, a
// question's tokens over a cached document).
// Each tile of 16 MFMA columns is (position, row) = (i / 8, i % 8) of two
// positions, and the fp16 hi and lo parts of the query and of P are stacked
// along the reductions (QK: the same decoded K against the hi and the lo
// query; PV: the hi and the lo P against the same decoded V), so each lane's
// column is one query row and its softmax runs once.  A unit of one position
// holds its rows' hi parts in columns 0-7 and lo parts in 8-15 instead: half
// the MFMAs.
// Eight waves of 32-token chunks per workgroup, one workgroup per CU (the
// decode tables).  PAGED: the grid is one workgroup per work segment of the
// step's plan (paged_plan_kernel).  Slot-mapped: grid (split, kv head, unit).
// D = 64: half the k-steps and PV tiles per token, the fp16 lo parts of V and
// turbo_prod's K and powers of two for the query rows and V, as
// dec::attn_decode_split_kernel.
// Issue-bound at many passes per workgroup (D = 128, 32 sequences of 1K-32K
// tokens: 94 us), bound by the setup and the merge at few.  A D = 64 step of
// 8 sequences (500-4,000 tokens, 2 new tokens, 2 heads) with its append takes
// 22.1 us, against 212.6 on the generic kernels it ran on before.
// ---------------------------------------------------------------------------
namespace unit {
using namespace mfma;
constexpr int kNP = 4;                // positions (row groups) per unit
constexpr int kNT = kNP / 2;          // tiles of 16 MFMA columns
constexpr int kWaves = 8, kChunk = 32, kPass = kWaves * kChunk;
constexpr int kTiles = kChunk / 16;   // QK tiles of a chunk
constexpr int kR = kRows * kNP;       // query rows of the workgroup
constexpr int kMoRows = 16;           // rows merged per tile
// Decode tables in the layout of decode_table_words: S rows at byte 0 and K|V
// rows at byte kOffKV.  One address reads a code byte's S pair (offset 0) and
// its K pair (offset kOffKV, which no two-address LDS read merges with 0),
// each straight into its MFMA operand; a V lookup's address is that of the
// byte's S row + 128 (turbo_prod's V copies; turbo_mse reads its K copies,
// + 0).  turbo_prod's V lo parts (D = 64) are copies of the S rows' upper
// halves, kLoCopies of them.  After the token loop the space holds the waves'
// results for the merge, one tile in each half.
constexpr int kOffKV = 65520;
constexpr int kTabWords = 32768;
constexpr int kLoCopies = 28;
static_assert(kOffKV + 256 * 256 <= 4 * kTabWords, "K|V rows");
static_assert(256 * 255 + 128 + 4 * kLoCopies <= kOffKV, "the V lo rows end below the K table");
static_assert(kRows % kWaves == 0 && kWaves == 8, "eight waves, one row per wave and position");
constexpr int part_stride(int D) { return D + 4; }  // paged partial row: o[D], m, l, pad
// A pass's weight in work positions: 4 for a unit of more than two positions
// (the two-tile loop), 3 otherwise, about their measured cost ratio.
__device__ __forceinline__ int pass_weight(int npos) { return npos > 2 ? 4 : 3; }
// Paged steps: the work positions a unit's setup counts for (a two-tile pass
// weighs 4), before its first pass (32 sequences of 1K-32K tokens: 139 us per
// step with 0, 135 with 4, 131-133 with 8, 12 or 16).
#ifndef TQ_PAGED_PIECE_COST
#define TQ_PAGED_PIECE_COST 8
#endif
constexpr int kPieceCost = TQ_PAGED_PIECE_COST;
// Row groups a split workgroup plans by itself (one wave, four groups per
// lane; the unit records take 16 bytes of LDS each).  Scans by DPP, divisions by
// the segment count through its inverse and the first unit found by the same wave
// took a small step's split kernel from 10.7 to 9.7 us.
constexpr int kPlanGroups = 256;
struct UnitRec {
    int32_t start, kv_end, seq;
    int16_t first, npos;
};

// The step's plan as paged_plan_kernel makes it, by one workgroup for itself:
// units in rec, then a sentinel; plan[0..2] = units, total work, segments per
// head.  Where the step has no more passes than Gh, every pass is a segment
// of its own (weight 1, no lead): no workgroup takes two while another has
// none, and the merge of a unit looks at its n passes instead of the segments
// they are scattered over; those segments go round the XCDs (seg = bl), the
// others are consecutive on each.  `scratch`: LDS of 2 (kPlanGroups + 8)
// words.  leave: write group_unit and plan for the merge.  Further results for
// workgroup bl of its head, in plan[3..6]: its segment, the segment's work
// positions [plan[4], plan[5]) (none: an empty segment), the unit holding the
// first of them.
__device__ __forceinline__ void plan_step(const PagedRows& pr, int num_rows, int max_kv_len, int Gh,
                                          int bl, bool leave, int* scratch, UnitRec* rec,
                                          int* plan) {
    const int groups = (num_rows + kRows - 1) / kRows;
    int* s_sq = scratch + 4;  // sequence of group g at [g], with room before and after
    int* s_gk = s_sq + kPlanGroups + 8;
    if (threadIdx.x < kPlanGroups) {
        // (unconditional loads: a group or row past the end re-reads the last)
        const int g = threadIdx.x, gc = min(g, groups - 1);
        int v[kRows];
        const int sq = pr.row_seq[(size_t)gc * kRows];
#pragma unroll
        for (int k = 0; k < kRows; ++k) v[k] = pr.row_kv_len[min(gc * kRows + k, num_rows - 1)];
        int m = 0;
#pragma unroll
        for (int k = 0; k < kRows; ++k)
            if (gc * kRows + k < num_rows) m = max(m, v[k]);
        s_sq[g] = sq;
        s_gk[g] = g < groups ? min(m, max_kv_len) : 0;
    }
    __syncthreads();
    // One group per lane, or four where there are more than 64.
    const auto plan_lanes = [&](auto per) {
        constexpr int P = decltype(per)::value;
        const int lane = threadIdx.x, g0 = P * lane;
        int sq[P + 4], gk[P + 3];  // sequences of groups g0 - 1 .. g0 + P + 2, lengths from g0
#pragma unroll
        for (int k = 0; k < P + 4; ++k) sq[k] = s_sq[min(max(g0 + k - 1, 0), kPlanGroups - 1)];
#pragma unroll
        for (int k = 0; k < P + 3; ++k) gk[k] = g0 + k < kPlanGroups ? s_gk[g0 + k] : 0;
        // The run each group is in: the last group at or before it that starts one.
        int last = -1;
#pragma unroll
        for (int k = 0; k < P; ++k)
            if (g0 + k < groups && (g0 + k == 0 || sq[k + 1] != sq[k])) last = g0 + k;
        const uint64_t below = __ballot(last >= 0) & ((1ull << lane) - 1ull);
        int cur = __shfl(last, below ? 63 - __clzll(below) : 0);
        int cnt[P], kv[P], n[P], lane_u = 0, lane_n = 0, lane_w = 0;
        bool start[P];
#pragma unroll
        for (int k = 0; k < P; ++k) {
            const int g = g0 + k;
            if (g < groups && (g == 0 || sq[k + 1] != sq[k])) cur = g;
            start[k] = g < groups && ((g - cur) & (kNP - 1)) == 0;
            cnt[k] = 1;
            kv[k] = gk[k];
#pragma unroll
            for (int m = 1; m < kNP; ++m)
                if (cnt[k] == m && g + m < groups && sq[k + 1 + m] == sq[k + 1]) {
                    ++cnt[k];
                    kv[k] = max(kv[k], gk[k + m]);
                }
            n[k] = start[k] ? (kv[k] + kPass - 1) / kPass : 0;
            lane_u += start[k] ? 1 : 0;
            lane_n += n[k];
            lane_w += n[k] > 0 ? kPieceCost + pass_weight(cnt[k]) * n[k] : 0;
        }
        const int su = wave_scan(lane_u), sn = wave_scan(lane_n), sw = wave_scan(lane_w);
        const int units = __builtin_amdgcn_readlane(su, 63);
        const int tn = __builtin_amdgcn_readlane(sn, 63), tw = __builtin_amdgcn_readlane(sw, 63);
        const bool single = tn <= Gh;
        const int total = single ? tn : tw, segs = single ? max(tn, 1) : Gh;
        const int seg = single ? bl : (bl & 7) * (Gh >> 3) + (bl >> 3);
        const Segments sg(total, segs, pr.inv_segments);
        const int b0 = seg < segs && total > 0 ? sg.bound(seg) : 0;
        const int b1 = seg < segs && total > 0 ? sg.bound(seg + 1) : 0;
        int u = su - lane_u, x = single ? sn - lane_n : sw - lane_w;
        int below_b0 = 0;  // units starting at or before b0
#pragma unroll
        for (int k = 0; k < P; ++k) {
            if (!start[k]) continue;
            const int w = single ? 1 : pass_weight(cnt[k]);
            x += !single && n[k] > 0 ? kPieceCost : 0;
            below_b0 += x <= b0 ? 1 : 0;
            rec[u] = UnitRec{x, kv[k], sq[k + 1], (int16_t)(g0 + k), (int16_t)cnt[k]};
            if (leave) {
#pragma unroll
                for (int m = 0; m < kNP; ++m)
                    if (m < cnt[k])
                        pr.group_unit[g0 + k + m] =
                            PagedUnit{g0 + k, cnt[k], kv[k], x, n[k], w, u, gk[k + m]};
            }
            x += w * n[k];
            ++u;
        }
        below_b0 = __builtin_amdgcn_readlane(wave_scan(below_b0), 63);
        if (lane == 0) {
            rec[units] = UnitRec{total, 0, 0, 0, 0};
            plan[0] = units;
            plan[1] = total;
            plan[2] = segs;
            plan[3] = seg;
            plan[4] = b0;
            plan[5] = b1;
            plan[6] = max(below_b0 - 1, 0);
            if (leave) {
                pr.plan[0] = units;
                pr.plan[1] = total;
                pr.plan[2] = segs;
            }
        }
    };
    if (threadIdx.x < 64) {
        if (groups <= 64)
            plan_lanes(std::integral_constant<int, 1>{});
        else
            plan_lanes(std::integral_constant<int, 4>{});
    }
    __syncthreads();
}

// A query or output row held by 16 lanes, so that a wave works on its row of
// all four positions at once instead of one after another.  Lane p owns elements 4j .. 4j + 3
// of the 64-element blocks, j = logical(p): in this order j ^ 1, j ^ 2, j ^ 4 and
// j ^ 8 are quad permutes, the half-row mirror and a row rotation, one DPP
// operand each: setup and merge of a unit of four, 2 passes, 16.0 -> 14.4 us;
// a step of 32 sequences (1.34 pieces per workgroup) 98.5 -> 96.0 us.
__device__ __forceinline__ int logical(int p) { return (p & 4) ? p ^ 3 : p; }
template <int M>
__device__ __forceinline__ float partner(float v) {  // v of logical lane j ^ M
    constexpr int ctrl = M == 1 ? 0xB1 : M == 2 ? 0x4E : M == 4 ? 0x141 : 0x128;
    static_assert(M == 1 || M == 2 || M == 4 || M == 8, "16 lanes");
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), ctrl, 0xF, 0xF, true));
}
// y[k] += c * (partner's y[k]) for 4 values (v_fmac_f32_dpp; the s_nop gives the
// two wait states a DPP read needs after the VALU write of its source).
#define TQ_FMAC4(CTRL)                                                          \
    asm("s_nop 1\n\t"                                                           \
        "v_fmac_f32_dpp %0, %0, %4 " CTRL " row_mask:0xf bank_mask:0xf\n\t"     \
        "v_fmac_f32_dpp %1, %1, %4 " CTRL " row_mask:0xf bank_mask:0xf\n\t"     \
        "v_fmac_f32_dpp %2, %2, %4 " CTRL " row_mask:0xf bank_mask:0xf\n\t"     \
        "v_fmac_f32_dpp %3, %3, %4 " CTRL " row_mask:0xf bank_mask:0xf"         \
        : "+v"(y[k]), "+v"(y[k + 1]), "+v"(y[k + 2]), "+v"(y[k + 3])            \
        : "v"(c))
template <int M, int E>
__device__ __forceinline__ void wht_across(float (&y)[E], int j) {
    const float c = (j & M) ? -1.0f : 1.0f;
#pragma unroll
    for (int k = 0; k < E; k += 4) {
        if constexpr (M == 1)
            TQ_FMAC4("quad_perm:[1,0,3,2]");
        else if constexpr (M == 2)
            TQ_FMAC4("quad_perm:[2,3,0,1]");
        else if constexpr (M == 4)
            TQ_FMAC4("row_half_mirror");
        else
            TQ_FMAC4("row_ror:8");
    }
}
#undef TQ_FMAC4
// Walsh-Hadamard transform of the row, left with a lane's sign
// (-1)^popcount(j) (each lane adds +-1 times its partner's value; both lanes of
// a pair carry the same sign).
template <int E>
__device__ __forceinline__ void wht_row16(float (&y)[E], int j) {
#pragma unroll
    for (int m = 1; m < E; m <<= 1)  // dims 1, 2 and (E = 8) 64
#pragma unroll
        for (int k = 0; k < E; ++k)
            if (!(k & m)) {
                const float a = y[k] + y[k + m], b = y[k] - y[k + m];
                y[k] = a;
                y[k + m] = b;
            }
    wht_across<1>(y, j);
    wht_across<2>(y, j);
    wht_across<4>(y, j);
    wht_across<8>(y, j);
}
__device__ __forceinline__ float lane_sign(int j) {
    return (__builtin_popcount(j & 15) & 1) ? -1.0f : 1.0f;
}

template <int SCH, int D, bool PAGED>
__global__ __launch_bounds__(64 * kWaves) void attn_unit_split_kernel(
    const uint16_t* __restrict__ query, const uint8_t* __restrict__ pool,
    const int32_t* __restrict__ slots, float* __restrict__ ws, float2* __restrict__ pml,
    uint16_t* __restrict__ output, float inv, int num_queries, int num_kv_tokens, int tokens_per_split, int num_splits, PageGeom g,
    PagedRows pr) {
    constexpr bool PROD = SCH == kSchProd;
    static_assert(SCH == kSchProd || SCH == kSchMse, "turbo_prod or turbo_mse pages");
    static_assert(D == 128 || D == 64, "head_dim 64 or 128");
    constexpr int kS = D / 32;   // QK k-steps; lane group gq holds dims [D/4 gq, D/4 gq + D/4)
    constexpr int kND = D / 16;  // PV tiles: lane i holds dims kND i .. + kND - 1
    constexpr int kE = D / 16;   // elements per lane of a row held by 16 lanes
    constexpr bool VLO = D == 64, QSCALE = D == 64, KLO = D == 64 && PROD;
    constexpr bool VSCALE = D == 64 || !PAGED;
    // MLO (turbo_mse): q's lo parts are stored x 2^kLoShift, so that their
    // product with K's hi parts and that of K's lo parts with q's hi parts share
    // an accumulator (cs).  KLO: the products with a lo part come first, while
    // the accumulator (cb) is small.  Added to a sum near the logit each costs a
    // rounding of it: logits of 20-85 were off by 7-8e-6 instead of 4.2-4.6e-6
    // (fp32 arithmetic: 3.9-4.8e-6).  With QSCALE log2(e) / sqrt(D) and the row's
    // power of two enter in the exponent's FMA, for the same reason.
    constexpr bool MLO = !PROD && (D == 64 || !PAGED);
    static_assert(kNT * sizeof(float) * kWaves * kMoRows * D <= 4 * kTabWords, "merge spaces");
    __shared__ __attribute__((aligned(256))) uint32_t lut[kTabWords];
    __shared__ uint4 bqs[kNP][kS][64];  // QK B operand (fp16 hi/lo q) of k-step s for lane l
    __shared__ uint64_t tko[kWaves][kChunk], tvo[kWaves][kChunk];
    __shared__ float4 tsc[kWaves][kChunk];  // per token: K scale a, residual scale b, vs / 2, bias
    __shared__ float mm[kWaves][kR], ml[kWaves][kR];
    __shared__ float rsc[QSCALE ? kR : 1];  // the rows' power of two

    // logit scale per unit ks (log2(e) / alpha folded at compile time: no run-time division)
    const float ck = inv * (PROD ? kLog2e / kAlphaK : kLog2e / kAlphaV);
    const float cr = inv * kLog2e;                                 // residual: ks * re
    // One work item: kv head h, row groups rg .. rg + npos - 1 (paged: of
    // sequence seq), tokens [t_begin, t_end) (paged: t_end is at most the unit's
    // longest row, and each row stops at its own length), partial slot pid
    // (slot-mapped: split pid).
    // (tid is a parameter so that a caller looping over items can keep the
    // per-thread values derived from it from being hoisted out of the loop
    // and held across the token loop.)
    auto item = [&](const int tid, const int h, const int rg, const int npos, const int seq,
                    const int t_begin, const int t_end, const size_t pid) {
        const int lane = tid & 63;
        const int w = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform (scalar)
        const int i = lane & 15, gq = lane >> 4;
        // Setup and merge: lane group gq holds the wave's row of position gq.
        const int j16 = logical(i);
        // Paged rows: per-row kv lengths (causal limit).  A piece past every
        // row's length has no partial (the combine does not read it).  Per
        // position: the group's longest row; per tile: this lane's column row
        // length; the shortest live row.
        int gend[kNP] = {}, rl_col[kNT] = {}, gmin_live = 0x7fffffff;
        const int ntile = (npos + 1) >> 1;  // tiles of 16 columns in use

        // A chunk's codes and per-token scales, loaded ahead of its compute.
        struct Chunk {
            uint32_t kw[kTiles][kS];  // K: tile tau, token 16*tau + i, bytes [4 kS gq, 4 kS gq + 4 kS)
            uint32_t vw[8];       // V: k-index 8gq + e (token below), bytes [D/32 i, D/32 i + D/32)
            uint16_t ks, re, vs;  // this lane's token's fp16 scales (raw: still in flight)
            bool valid;
        };
        // Token of this lane in the chunk at t0 (lanes past the range re-read the
        // last token of the range) and its slot, or for paged rows its page
        // table entry.  The load is issued here and consumed by fetch, so other
        // work runs in between; arithmetic on the loaded value here would make
        // the in-order vector-memory counter wait, right after the next chunk's
        // code loads are issued, for all of them (129-130 -> 125-127.5 us per
        // 32-sequence step).
        auto chunk_token = [&](int t0) -> int {
            return max(min(t0 + (lane & (kChunk - 1)), t_end - 1), 0);
        };
        auto load_slot = [&](int t0) -> int {
            const int t = chunk_token(t0);
            if constexpr (PAGED) {  // token t of sequence seq: page table entry t / B
                const int blk = g.bs_shift >= 0 ? t >> g.bs_shift : t / g.block_size;
                return pr.block_tables[(size_t)seq * pr.max_blocks + min(blk, pr.max_blocks - 1)];
            } else {
                return slots[t];
            }
        };
        // Token -> cell addresses (exchanged through LDS) -> scale and code
        // loads, issued for every lane; they stay in flight until the chunk is
        // computed.  Plain loads (not non-temporal): the workgroups of the two
        // kv heads of a work segment read each 128-byte code line together, one
        // through the other's L2 copy, and the units over one slot map read the
        // same cells.
        typedef __attribute__((address_space(1))) const uint8_t gbyte;
        typedef __attribute__((address_space(1))) const uint16_t ghalf;
        typedef __attribute__((address_space(1))) const uint32_t gword;
        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
        typedef __attribute__((address_space(1))) const u32x2 gpair;
        typedef __attribute__((address_space(1))) const u32x4 gquad;
        auto fetch = [&](int t0, int loaded, Chunk& c) {
            c.valid = t0 + (lane & (kChunk - 1)) < t_end && loaded >= 0;
            if constexpr (PAGED) {
                // loaded: the token's page table entry.  A cell's bytes are its
                // page's address plus 32-bit offsets within the page (integer
                // selects: no branches around loads).  Masked lanes (past the
                // range, or an unmapped page) address the workspace's spare page
                // instead: always valid memory, its bytes unused (bias -inf).
                const int t = chunk_token(t0);
                const int tib = g.bs_shift >= 0 ? t & (g.block_size - 1) : t % g.block_size;
                const uint32_t cell = (uint32_t)(tib * g.H + h);
                const uint8_t* pg =
                    c.valid ? pool + (uint64_t)(uint32_t)loaded * (uint32_t)g.page_size
                            : pr.spare_page;
                const uint32_t so = cell * (uint32_t)g.scale_stride;
                c.ks = ld_u16(pg + (so + (uint32_t)g.ks_off));
                c.vs = ld_u16(pg + (so + (uint32_t)g.vs_off));
                c.re = PROD ? ld_u16(pg + (so + (uint32_t)g.kres_off)) : (uint16_t)0;
                const uint32_t co = cell * (uint32_t)g.code_stride;
                tko[w][lane & (kChunk - 1)] = reinterpret_cast<uint64_t>(pg + (co + (uint32_t)g.kc_off));
                tvo[w][lane & (kChunk - 1)] = reinterpret_cast<uint64_t>(pg + (co + (uint32_t)g.vc_off));
            } else {
                // loaded: the token's slot.  Masked lanes (past the range, or a
                // negative slot) read the first bytes of the query instead.
                int page, tib;
                split_slot(c.valid ? loaded : 0, g, page, tib);
                const uint64_t cell = (uint64_t)(tib * g.H + h);
                const uint8_t* pg = pool + (uint64_t)page * g.page_size;
                const uint8_t* dummy = reinterpret_cast<const uint8_t*>(query);
                const uint64_t so = cell * g.scale_stride, co = cell * g.code_stride;
                c.ks = ld_u16(c.valid ? pg + (so + g.ks_off) : dummy);
                c.vs = ld_u16(c.valid ? pg + (so + g.vs_off) : dummy + 2);
                c.re = PROD ? ld_u16(c.valid ? pg + (so + g.kres_off) : dummy + 4) : (uint16_t)0;
                tko[w][lane & (kChunk - 1)] =
                    reinterpret_cast<uint64_t>(c.valid ? pg + (co + g.kc_off) : dummy);
                tvo[w][lane & (kChunk - 1)] =
                    reinterpret_cast<uint64_t>(c.valid ? pg + (co + g.vc_off) : dummy);
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int tau = 0; tau < kTiles; ++tau) {
                gbyte* kp = reinterpret_cast<gbyte*>(tko[w][16 * tau + i]) + 4 * kS * gq;
                if constexpr (D == 128) {
                    const u32x4 x = *reinterpret_cast<gquad*>(kp);
#pragma unroll
                    for (int s = 0; s < kS; ++s) c.kw[tau][s] = x[s];
                } else {
                    const u32x2 x = *reinterpret_cast<gpair*>(kp);
#pragma unroll
                    for (int s = 0; s < kS; ++s) c.kw[tau][s] = x[s];
                }
            }
            // (the K words first: the QK waits for them while the V words may
            // still be in flight)
            __builtin_amdgcn_sched_barrier(0);
            // k-index 8gq + e is token 4gq + e (e < 4) or 16 + 4gq + (e - 4).
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int tok = e < 4 ? 4 * gq + e : 16 + 4 * gq + (e - 4);
                gbyte* vp = reinterpret_cast<gbyte*>(tvo[w][tok]) + D / 32 * i;
                if constexpr (D == 128)
                    c.vw[e] = *reinterpret_cast<gword*>(vp);
                else
                    c.vw[e] = *reinterpret_cast<ghalf*>(vp);
            }
        };

        // Issue order matters (the vector-memory counter is in order): the first
        // chunk's slots, which the code loads wait for; this wave's query rows
        // (row r of the workgroup is row r % 8 of group rg + r / 8: rows rg * 8 +
        // r); paged rows' lengths, which nothing needs before the codes are out.
        // (The unit's sequence and end come with the plan: read here before the
        // slots, they were one more memory latency ahead of every piece.)
        int t0 = t_begin + w * kChunk;
        const int slot0 = load_slot(t0);
        uint32_t qraw[kE / 2];
        {
            const int qi = min(rg * kRows + w + gq * kWaves, num_queries - 1);
            const uint32_t* qp = reinterpret_cast<const uint32_t*>(
                query + ((size_t)qi * g.H + h) * D + 4 * j16);
#pragma unroll
            for (int k = 0; k < kE / 2; ++k) qraw[k] = qp[(k & 1) + 32 * (k >> 1)];
        }
        // (every length unconditionally, rows past the end re-read the last
        // row: a load under a condition sits in a branch whose join waits for it)
        int lraw[kNP];
        if constexpr (PAGED) {
#pragma unroll
            for (int p = 0; p < kNP; ++p)
                lraw[p] = pr.row_kv_len[min((rg + p) * kRows + (lane & 7), num_queries - 1)];
        }
        __builtin_amdgcn_sched_barrier(0);
        // Query halves to fp32 (times the sign flip) before the code loads are
        // issued, so waiting for them never waits for the codes.
        float qf[kE];
        {
            const float sh = (h & 1) ? -1.0f : 1.0f;
#pragma unroll
            for (int k = 0; k < kE; k += 2) {
                qf[k] = h2f(qraw[k / 2] & 0xffff) * sh;
                qf[k + 1] = h2f(qraw[k / 2] >> 16) * (-sh);
            }
        }
        Chunk cur;
        fetch(t0, slot0, cur);  // in flight during the setup below (empty waves: all invalid)
        __builtin_amdgcn_sched_barrier(0);  // the first chunk's loads go out before the setup
        if constexpr (PAGED) {
#pragma unroll
            for (int p = 0; p < kNP; ++p) {
                const int rr = (rg + p) * kRows + (lane & 7);
                const int lv = p < npos && rr < num_queries ? lraw[p] : 0;
                // column i's row of position p is row i % 8 = lane % 8
                // (one position: both halves of the tile hold its rows, hi and lo)
                if (npos == 1 ? p == 0 : (i >> 3) == (p & 1)) rl_col[p >> 1] = lv;
                // over the 8 rows: lane ^ 1, ^ 2, then 7 - lane of each 8
                int m = lv, n = lv;
                const auto over = [&](auto ctrl) {
                    m = max(m, __builtin_amdgcn_mov_dpp(m, decltype(ctrl)::value, 0xF, 0xF, true));
                    n = min(n, __builtin_amdgcn_mov_dpp(n, decltype(ctrl)::value, 0xF, 0xF, true));
                };
                over(std::integral_constant<int, 0xB1>{});
                over(std::integral_constant<int, 0x4E>{});
                over(std::integral_constant<int, 0x141>{});
                gend[p] = __builtin_amdgcn_readfirstlane(m);
                const int gmin = __builtin_amdgcn_readfirstlane(n);
                if (p < npos) gmin_live = min(gmin_live, gmin);
            }
        }
        // The decode tables from registers, and each wave's rotated rows (lane
        // group k: row w of group rg + k) as fp16 hi and lo parts straight into
        // the QK B operand: one barrier for the setup.  A lane's dims 4j .. 4j + 3
        // (and 64 + 4j ..) lie in k-group d / (8 kS), k-step (j / 2) % kS, halves
        // 4(j % 2) .. of the half8.  Two or more positions: tile k / 2, column
        // 8(k % 2) + w, hi in operand 2(k / 2), lo in 2(k / 2) + 1; one position:
        // tile 0, hi in column w, lo in column w + 8.
        {
            const TableWords<PROD> tw = decode_table_words<PROD, KLO>(w, lane);
            wht_row16(qf, j16);
            const bool live = gq < npos && rg * kRows + w + gq * kWaves < num_queries;
            const float qs = live ? inv * lane_sign(j16) : 0.0f;
#pragma unroll
            for (int k = 0; k < kE; ++k) qf[k] = live ? qf[k] * qs : 0.0f;
            if constexpr (QSCALE) {
                float m = 0.0f;
#pragma unroll
                for (int k = 0; k < kE; ++k) m = fmaxf(m, fabsf(qf[k]));
                m = fmaxf(m, partner<1>(m));
                m = fmaxf(m, partner<2>(m));
                m = fmaxf(m, partner<4>(m));
                m = fmaxf(m, partner<8>(m));
                const int ex = scale_exp(m);
#pragma unroll
                for (int k = 0; k < kE; ++k) qf[k] = __builtin_amdgcn_ldexpf(qf[k], -ex);
                if (i == 0) rsc[gq * kRows + w] = __builtin_amdgcn_ldexpf(1.0f, ex);
            }
            if (npos == 1 ? gq == 0 : gq < 2 * ntile) {  // (the other rows are never read)
                const int col_hi = npos == 1 ? w : 8 * (gq & 1) + w;
                const int col_lo = npos == 1 ? w + 8 : col_hi;
                const int op_hi = npos == 1 ? 0 : 2 * (gq >> 1);
                const int op_lo = npos == 1 ? 0 : op_hi + 1;
                const int s_l = (j16 >> 1) & (kS - 1), g_l = j16 / (2 * kS);
#pragma unroll
                for (int k = 0; k < kE; k += 4) {
                    const uint32_t h0 = pack_h2(qf[k], qf[k + 1]), h1 = pack_h2(qf[k + 2], qf[k + 3]);
                    const int at = 16 * (g_l + k / 2);  // (second block: two k-groups on)
                    reinterpret_cast<uint2*>(&bqs[op_hi][s_l][at + col_hi])[j16 & 1] =
                        make_uint2(h0, h1);
                    uint2 lo = make_uint2(lo_pair(qf[k], qf[k + 1], h0), lo_pair(qf[k + 2], qf[k + 3], h1));
                    if (MLO && npos > 1)
                        lo = make_uint2(pack_h2(lo_part(qf[k]), lo_part(qf[k + 1])),
                                        pack_h2(lo_part(qf[k + 2]), lo_part(qf[k + 3])));
                    reinterpret_cast<uint2*>(&bqs[op_lo][s_l][at + col_lo])[j16 & 1] = lo;
                }
            }
            store_decode_tables<PROD>(lut, kOffKV / 4, w, lane, tw);
            if constexpr (VLO && PROD) {
                uint32_t vlo[4];
                lo_table_words(w, lane, vlo);
                if ((lane & 7) < kLoCopies / 4) {
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        *reinterpret_cast<u32x4*>(
                            &lut[(32 * w + 8 * k + (lane >> 3)) * 64 + 32 + 4 * (lane & 7)]) =
                            (u32x4){vlo[k], vlo[k], vlo[k], vlo[k]};
                }
            }
        }
        lds_barrier();
        // The S-row address of byte b of word (this lane's copy; its K pair at
        // + kOffKV), and that of a V code byte (S row + 128: its V pair at
        // + kOffKV): the code byte goes into byte 1 (entry stride 256 B) with one
        // v_perm, byte 1 of the base is re-added.
        const uint32_t luts = (uint32_t)reinterpret_cast<uintptr_t>((lds_u32*)&lut[lane & 31]);
        const uint32_t luts_hi = luts & 0xFF00u;
        auto s_addr = [&](uint32_t word, int b, uint32_t off) -> uint32_t {
            return __builtin_amdgcn_perm(word, luts + off, 0x03020000u | ((4u + b) << 8)) + luts_hi;
        };
        auto lds_at = [](uint32_t a, int off) -> uint32_t {
            return *reinterpret_cast<const lds_u32*>(a + off);
        };
        // V lookups' offset from the S row; with VLO the lanes past the lo
        // copies read their copy kLoCopies below.
        const uint32_t voff = !PROD ? 0u
                              : VLO && (lane & 31) >= kLoCopies ? 128u - 4u * kLoCopies
                                                                : 128u;

        int slot_nx = load_slot(t0 + kPass);
        // One softmax state per lane and tile (its column's row; m_col: the
        // reference, k below the maximum), hi and lo
        // stacked along the reductions.  A unit with fewer positions runs the
        // loop over the tiles it needs; a tile's unused columns compute on zero
        // queries and are dropped.
        float m_col[kNT], l_col[kNT];
        f32x4 acc_col[kNT][kND], acl_col[VLO ? kNT : 1][VLO ? kND : 1];
#pragma unroll
        for (int t = 0; t < kNT; ++t) {
            m_col[t] = kInitMax;
            l_col[t] = 0.0f;
#pragma unroll
            for (int v = 0; v < kND; ++v) {
                acc_col[t][v] = (f32x4){0.f, 0.f, 0.f, 0.f};
                if constexpr (VLO) acl_col[t][v] = (f32x4){0.f, 0.f, 0.f, 0.f};
            }
        }
        VPower vp;  // VSCALE
        float qsc[kNT];
#pragma unroll
        for (int t = 0; t < kNT; ++t)
            qsc[t] = QSCALE && t < ntile ? ck * rsc[npos == 1 ? i & 7 : 16 * t + i] : 1.0f;
        // COLS (a unit of one position): one tile whose columns are the
        // position's rows as hi (columns 0-7) and lo (8-15) parts: one MFMA per
        // product instead of two, and the two halves of a column pair summed
        // (logits; outputs at the merge).
        auto stacked_loop = [&](auto nta, auto cols) {
            constexpr int NTA = decltype(nta)::value;
            constexpr bool COLS = decltype(cols)::value;
            static_assert(!COLS || NTA == 1, "one tile");
            while (t0 < t_end) {  // wave-uniform
                const float k_old = vp.k;
                if constexpr (VSCALE) vp.raise(cur.valid ? cur.vs : 0u);
                {
                    const float ks = h2f(cur.ks), vs = h2f(cur.vs), re = PROD ? h2f(cur.re) : 0.0f;
                    const float kx = QSCALE ? 1.0f : ck, kr = QSCALE ? kAlphaK : cr;
                    tsc[w][lane & (kChunk - 1)] =
                        cur.valid ? make_float4(ks * kx,
                                                PROD  ? ks * re * kr
                                                : MLO ? low_factor(ks * kx)
                                                      : ks * kx * kLoScale,
                                                0.5f * vs, 0.0f)
                                  : make_float4(0.f, 0.f, 0.f, -INFINITY);
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                const int t1 = t0 + kPass;
                // QK: each decoded A operand against every tile's hi and lo query
                f32x4 cb[NTA][kTiles], cs[NTA][kTiles];
#pragma unroll
                for (int tau = 0; tau < kTiles; ++tau)
#pragma unroll
                    for (int t = 0; t < NTA; ++t) {
                        cb[t][tau] = (f32x4){0.f, 0.f, 0.f, 0.f};
                        cs[t][tau] = cb[t][tau];
                    }
                // The operands of k-step s + 1 (query parts, decoded codes) are
                // read from LDS before the MFMAs of step s.
                struct Ops {
                    half8 bk[2 * NTA];  // k-step s of each tile's hi and lo query
                    half8 a[kTiles], al[kTiles];
                };
                auto load_ops = [&](int s, Ops& o) {
#pragma unroll
                    for (int pp = 0; pp < (COLS ? 1 : 2 * NTA); ++pp)
                        o.bk[pp] = __builtin_bit_cast(half8, bqs[pp][s][lane]);
#pragma unroll
                    for (int tau = 0; tau < kTiles; ++tau) {
                        // one address per byte: its K pair (prod aK*K3, mse the hi
                        // parts) and its S pair (prod the residual signs, mse the lo
                        // parts)
                        uint32_t ad[4];
#pragma unroll
                        for (int b = 0; b < 4; ++b) ad[b] = s_addr(cur.kw[tau][s], b, 0);
                        o.a[tau] = as_h8(lds_at(ad[0], kOffKV), lds_at(ad[1], kOffKV),
                                         lds_at(ad[2], kOffKV), lds_at(ad[3], kOffKV));
                        o.al[tau] = as_h8(lds_at(ad[0], 0), lds_at(ad[1], 0), lds_at(ad[2], 0),
                                          lds_at(ad[3], 0));
                    }
                };
                Ops ops[2];
                float4 scq[kTiles][4];  // the logits' per-token scales, read during the last k-step
                load_ops(0, ops[0]);
#pragma unroll
                for (int s = 0; s < kS; ++s) {
                    if (s < kS - 1) {
                        load_ops(s + 1, ops[(s + 1) & 1]);
                    } else {
#pragma unroll
                        for (int tau = 0; tau < kTiles; ++tau)
#pragma unroll
                            for (int e = 0; e < 4; ++e) scq[tau][e] = tsc[w][16 * tau + 4 * gq + e];
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    const Ops& o = ops[s & 1];
#pragma unroll
                    for (int tau = 0; tau < kTiles; ++tau) {
#pragma unroll
                        for (int t = 0; t < NTA; ++t) {
                            if constexpr (!KLO) cb[t][tau] = mma(o.a[tau], o.bk[2 * t], cb[t][tau]);
                            if constexpr (!COLS) {
                                f32x4& c = MLO ? cs[t][tau] : cb[t][tau];
                                c = mma(o.a[tau], o.bk[2 * t + 1], c);
                            }
                        }
                        // prod: the +-1 residual signs against the hi and lo query;
                        // mse: the codebook's lo parts (into cs) against the hi query
                        // only: the product of the two lo parts, each below 2^-11
                        // of its value, is at most 2^-22 of the logit's terms (KLO: so
                        // K's lo parts, into cb)
                        half8 sg = o.al[tau];
                        if constexpr (KLO) {
#pragma unroll
                            for (int t = 0; t < NTA; ++t)
                                cb[t][tau] = mma(o.al[tau], o.bk[2 * t], cb[t][tau]);
                            sg = sign_octet(cur.kw[tau][s]);
                        }
#pragma unroll
                        for (int t = 0; t < NTA; ++t) {
                            cs[t][tau] = mma(sg, o.bk[2 * t], cs[t][tau]);
                            if (!COLS && PROD) cs[t][tau] = mma(sg, o.bk[2 * t + 1], cs[t][tau]);
                        }
                    }
                    if constexpr (KLO) {
                        static_assert(kS == 2, "both k-steps' operands in ops");
                        if (s == kS - 1)
#pragma unroll
                            for (int k = 0; k < kS; ++k)
#pragma unroll
                                for (int tau = 0; tau < kTiles; ++tau)
#pragma unroll
                                    for (int t = 0; t < NTA; ++t)
                                        cb[t][tau] = mma(ops[k].a[tau], ops[k].bk[2 * t], cb[t][tau]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                // Logits (base 2; QSCALE: before their row's factor qsc) of tokens
                // 16*tau + 4*gq + e for this lane's column.
                float lg[NTA][kTiles][4];
#pragma unroll
                for (int t = 0; t < NTA; ++t)
#pragma unroll
                    for (int tau = 0; tau < kTiles; ++tau)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float4 sc = scq[tau][e];
                            float b = cb[t][tau][e], r = cs[t][tau][e];
                            float low = 0.0f;
                            if constexpr (COLS) {  // + the partner column (lane ^ 8)
                                const float p = lane_xor<8>(b);
                                const float lo = i & 8 ? b : p;
                                r += lane_xor<8>(r);
                                if constexpr (QSCALE && !PROD) r = fmaf(lo, (float)(1 << kLoShift), r);
                                low = fmaf(r, sc.y, sc.w);
                                if constexpr (QSCALE && PROD) low = fmaf(lo, sc.x, low);
                                b = !QSCALE ? b + p : i & 8 ? p : b;
                            } else {
                                low = fmaf(r, sc.y, sc.w);
                            }
                            lg[t][tau][e] = fmaf(b, sc.x, low);
                        }
                // The V lookups (B operands of PV) go out before the softmax,
                // whose VALU work hides their LDS latency.
                uint32_t bv[kND][4], bl[VLO ? kND : 1][4];  // [N-tile v = d - kND i][token pair]
                if constexpr (D == 128) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const uint32_t we = cur.vw[2 * q], wo = cur.vw[2 * q + 1];
                        const uint32_t lob = (we & 0x0F0F0F0Fu) | ((wo & 0x0F0F0F0Fu) << 4);
                        const uint32_t hib = ((we >> 4) & 0x0F0F0F0Fu) | (wo & 0xF0F0F0F0u);
#pragma unroll
                        for (int b = 0; b < 4; ++b) {
                            // (turbo_prod: the V copies; turbo_mse: its K copies hold aV*V4)
                            bv[2 * b][q] = lds_at(s_addr(lob, b, PROD ? 128u : 0u), kOffKV);
                            bv[2 * b + 1][q] = lds_at(s_addr(hib, b, PROD ? 128u : 0u), kOffKV);
                        }
                    }
                } else {
                    // two token pairs per word (a lane's row part is two bytes)
#pragma unroll
                    for (int p = 0; p < 2; ++p) {
                        const uint32_t we = cur.vw[4 * p] | (cur.vw[4 * p + 2] << 16);
                        const uint32_t wo = cur.vw[4 * p + 1] | (cur.vw[4 * p + 3] << 16);
                        const uint32_t lob = (we & 0x0F0F0F0Fu) | ((wo & 0x0F0F0F0Fu) << 4);
                        const uint32_t hib = ((we >> 4) & 0x0F0F0F0Fu) | (wo & 0xF0F0F0F0u);
#pragma unroll
                        for (int b = 0; b < 4; ++b) {
                            const int v = 2 * (b & 1), q = 2 * p + (b >> 1);
                            const uint32_t a0 = s_addr(lob, b, voff), a1 = s_addr(hib, b, voff);
                            bv[v][q] = lds_at(a0, kOffKV);
                            bv[v + 1][q] = lds_at(a1, kOffKV);
                            if constexpr (VLO) {
                                bl[v][q] = lds_at(a0, 0);
                                bl[v + 1][q] = lds_at(a1, 0);
                            }
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
                // This chunk's codes are consumed: the next chunk's codes and the
                // slots of the one after are fetched into cur's registers, in
                // flight during the softmax and PV (no copy at the end of the
                // step, which would wait for them: 128.3 -> 127.1 us turbo_prod,
                // 129.5 -> 127.1 us turbo_mse against fetching into a second
                // buffer behind the first k-step).
                if (t1 < t_end) {
                    fetch(t1, slot_nx, cur);
                    slot_nx = load_slot(t1 + kPass);
                }
                const bool row_ends = PAGED && t0 + kChunk > gmin_live;
                if (row_ends) {  // a row of the unit ends in this chunk
                    // (wave-uniform; a branch: no selects on every chunk)
                    asm volatile("" ::: "memory");
#pragma unroll
                    for (int t = 0; t < NTA; ++t)
#pragma unroll
                        for (int tau = 0; tau < kTiles; ++tau)
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                if (t0 + 16 * tau + 4 * gq + e >= rl_col[t])
                                    lg[t][tau][e] = -INFINITY;
                }
                // Online softmax with a lagging maximum: m_col moves (and the
                // accumulators are rescaled) only when a logit passes it by more
                // than 1, so the weights stay <= 2 (2^(k + 1)): the PV operand is
                // P * vs / 2.
                float mloc[NTA];
                bool grow = VSCALE && vp.k != k_old;
#pragma unroll
                for (int t = 0; t < NTA; ++t) {
                    // (IEEE maximum: no canonicalising of the lane-exchanged
                    // values; a NaN logit leaves grow false, as fmaxf would)
                    float m = lg[t][0][0];
#pragma unroll
                    for (int k = 1; k < 4 * kTiles; ++k)
                        m = __builtin_elementwise_maximum(m, lg[t][k >> 2][k & 3]);
                    const auto mx = [](float x, float y) { return __builtin_elementwise_maximum(x, y); };
                    m = lane_xor_reduce<16>(m, mx);
                    mloc[t] = lane_xor_reduce<32>(m, mx) * (QSCALE ? qsc[t] : 1.0f);
                    grow = grow || (VSCALE ? mloc[t] - vp.k : mloc[t]) > m_col[t] + 1.0f;
                }
                if (__any(grow)) {  // wave-uniform
#pragma unroll
                    for (int t = 0; t < NTA; ++t) {
                        const float m_new = VSCALE ? fmaxf(m_col[t] + k_old, mloc[t]) - vp.k
                                                   : fmaxf(m_col[t], mloc[t]);
                        const float alpha = __builtin_amdgcn_exp2f(m_col[t] - m_new);
                        m_col[t] = m_new;
                        l_col[t] *= alpha;
                        // acc lane (d, gq) holds rows 4gq .. 4gq + 3 (columns of lanes 4gq + e)
                        float a[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) a[e] = __shfl(alpha, 4 * gq + e);
#pragma unroll
                        for (int v = 0; v < kND; ++v)
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                acc_col[t][v][e] *= a[e];
                                if constexpr (VLO) acl_col[t][v][e] *= a[e];
                            }
                    }
                }
#pragma unroll
                for (int t = 0; t < NTA; ++t) {
#pragma unroll
                    for (int tau = 0; tau < kTiles; ++tau)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            lg[t][tau][e] = __builtin_amdgcn_exp2f(
                                QSCALE ? fmaf(lg[t][tau][e], qsc[t], -m_col[t]) : lg[t][tau][e] - m_col[t]);
                    // pairwise: no zero start, and the adds do not wait on one another
                    float part[kTiles];
#pragma unroll
                    for (int tau = 0; tau < kTiles; ++tau)
                        part[tau] = (lg[t][tau][0] + lg[t][tau][1]) + (lg[t][tau][2] + lg[t][tau][3]);
                    float lsum = part[0];
#pragma unroll
                    for (int tau = 1; tau < kTiles; ++tau) lsum += part[tau];
                    l_col[t] += lsum;
                }
                // PV: every tile's hi and lo P against each decoded B operand
                half8 ah[NTA], al[NTA];
#pragma unroll
                for (int t = 0; t < NTA; ++t)
#pragma unroll
                    for (int tau = 0; tau < kTiles; ++tau)
#pragma unroll
                        for (int e = 0; e < 4; ++e) lg[t][tau][e] *= tsc[w][16 * tau + 4 * gq + e].z;
                if (row_ends) {
                    // a token past the column's row: 0 also where its V scale is
                    // infinite or NaN (0 times it is NaN)
                    asm volatile("" ::: "memory");
#pragma unroll
                    for (int t = 0; t < NTA; ++t)
#pragma unroll
                        for (int tau = 0; tau < kTiles; ++tau)
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                if (t0 + 16 * tau + 4 * gq + e >= rl_col[t]) lg[t][tau][e] = 0.0f;
                }
#pragma unroll
                for (int t = 0; t < NTA; ++t) {
                    uint32_t hw[4], lw[4];
#pragma unroll
                    for (int e = 0; e < 8; e += 2) {
                        const float x0 = lg[t][e >> 2][e & 3], x1 = lg[t][e >> 2][(e & 3) + 1];
                        hw[e >> 1] = pack_h2(x0, x1);
                        lw[e >> 1] = lo_pair(x0, x1, hw[e >> 1]);
                    }
                    if constexpr (COLS) {  // column i < 8: hi; i >= 8: lo
                        const bool lo = (i >> 3) != 0;
                        ah[t] = as_h8(lo ? lw[0] : hw[0], lo ? lw[1] : hw[1], lo ? lw[2] : hw[2],
                                      lo ? lw[3] : hw[3]);
                    } else {
                        ah[t] = as_h8(hw[0], hw[1], hw[2], hw[3]);
                        al[t] = as_h8(lw[0], lw[1], lw[2], lw[3]);
                    }
                }
#pragma unroll
                for (int v = 0; v < kND; ++v) {
                    const half8 bvv = as_h8(bv[v][0], bv[v][1], bv[v][2], bv[v][3]);
#pragma unroll
                    for (int t = 0; t < NTA; ++t) {
                        acc_col[t][v] = mma(ah[t], bvv, acc_col[t][v]);
                        if (!COLS) acc_col[t][v] = mma(al[t], bvv, acc_col[t][v]);
                    }
                }
                if constexpr (VLO) {  // (the lo P against V's lo parts: ~2^-22 of the sum, left out)
#pragma unroll
                    for (int v = 0; v < kND; ++v) {
                        const half8 blv = as_h8(bl[v][0], bl[v][1], bl[v][2], bl[v][3]);
#pragma unroll
                        for (int t = 0; t < NTA; ++t) acl_col[t][v] = mma(ah[t], blv, acl_col[t][v]);
                    }
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                t0 = t1;
            }
        };
        if (ntile == 2)
            stacked_loop(std::integral_constant<int, 2>{}, std::false_type{});
        else if (npos == 1)
            stacked_loop(std::integral_constant<int, 1>{}, std::true_type{});
        else
            stacked_loop(std::integral_constant<int, 1>{}, std::false_type{});

        // Wave results: l summed over the g lanes of each column; o rows with
        // the V codebook scale divided out.  Then the waves are merged per row,
        // the inverse WHT and sign flip applied, and the partial written.  A
        // position whose rows all end before this piece has no partial (its
        // combine reads only the pieces below its longest row).
#pragma unroll
        for (int t = 0; t < kNT; ++t) {
            float l_tot = lane_xor_reduce<16>(l_col[t], [](float x, float y) { return x + y; });
            l_tot = lane_xor_reduce<32>(l_tot, [](float x, float y) { return x + y; });
            if (gq == 0) {
                mm[w][16 * t + i] = m_col[t];
                ml[w][16 * t + i] = l_tot;
            }
        }
        const float iav = 1.0f / kAlphaV;
        // Both tiles at once, tile t's merge space at table word 16384 t (the
        // tables are no longer read).  Then wave w merges row w of every
        // position: lane group gq the waves' (m, l, o) of position gq, elements
        // 4j .. 4j + 3 (and 64 + 4j ..) per lane, then the inverse WHT and sign
        // flip, and the partial.
        auto mot = [&](int t) { return reinterpret_cast<float(*)[kMoRows][D]>(&lut[16384 * t]); };
        __syncthreads();  // every wave is done with the tables
#pragma unroll
        for (int t = 0; t < kNT; ++t) {
            if (t >= ntile) break;  // wave- and workgroup-uniform
#pragma unroll
            for (int v = 0; v < kND; ++v)
#pragma unroll
                for (int e = 0; e < 4; ++e) {  // (x2: the PV operand was P * vs / 2)
                    float x = acc_col[t][v][e];
                    if constexpr (VLO) x = fmaf(acl_col[t][v][e], kLoScale, x);
                    mot(t)[w][4 * gq + e][kND * i + v] = x * (2.0f * iav);
                }
        }
        __syncthreads();
        {
            const int rr = 8 * (gq & 1) + w;  // this lane group's row of its tile
            const int r = kMoRows * (gq >> 1) + rr;
            // (a unit of one position: group 1 holds the same rows' lo columns;
            // with one tile, groups 2 and 3 merge tile 0's rows and drop them)
            const float(*mt)[kMoRows][D] = mot(ntile == 2 ? gq >> 1 : 0);
            float pm[kWaves], pl[kWaves];
#pragma unroll
            for (int u = 0; u < kWaves; ++u) pm[u] = mm[u][r], pl[u] = ml[u][r];
            float M = pm[0];
#pragma unroll
            for (int u = 1; u < kWaves; ++u) M = fmaxf(M, pm[u]);
            float L = 0.f, o[kE];
#pragma unroll
            for (int k = 0; k < kE; ++k) o[k] = 0.f;
#pragma unroll
            for (int u = 0; u < kWaves; ++u) {
                const float wt = __builtin_amdgcn_exp2f(pm[u] - M);  // (argument <= 0)
                L += pl[u] * wt;
#pragma unroll
                for (int k = 0; k < kE; k += 4) {
                    const float4 x = *reinterpret_cast<const float4*>(&mt[u][rr][4 * j16 + 16 * k]);
                    o[k] += x.x * wt;
                    o[k + 1] += x.y * wt;
                    o[k + 2] += x.z * wt;
                    o[k + 3] += x.w * wt;
                }
            }
            if (npos == 1) {  // + the lo columns (wave-uniform)
#pragma unroll
                for (int k = 0; k < kE; ++k) o[k] += lane_xor<16>(o[k]);
            }
            wht_row16(o, j16);
            const float s0 = ((h & 1) ? -inv : inv) * lane_sign(j16);
            bool keep = gq < npos;
            if constexpr (PAGED)
                keep = keep && t_begin < (gq == 0 ? gend[0] : gq == 1 ? gend[1] : gq == 2 ? gend[2] : gend[3]);
            else
                keep = keep && rg * kRows + r < num_queries;
            // paged: rows of part_stride with (m, l) behind them; slot-mapped:
            // the layout of dec's partials (attn_decode_combine_kernel)
            const size_t it = (size_t)(rg + gq) * g.H + h;
            float* po = PAGED ? ws + ((pid * kNP + gq) * kRows + w) * part_stride(D)
                              : ws + ((it * num_splits + pid) * kRows + w) * D;
            float2* pm2 = PAGED ? reinterpret_cast<float2*>(po + D)
                                : pml + (it * kRows + w) * num_splits + pid;
            if (!PAGED && num_splits == 1) {  // nothing to merge: the output itself
                uint16_t* out = output + ((size_t)(rg * kRows + r) * g.H + h) * D + 4 * j16;
                const auto fin = [&](float x) { return (uint32_t)f2h(L > 0.f ? x / L : x); };
                if (keep) {
#pragma unroll
                    for (int k = 0; k < kE; k += 4)
                        store_h4(out + 16 * k, fin(o[k] * s0) | (fin(o[k + 1] * -s0) << 16),
                                 fin(o[k + 2] * s0) | (fin(o[k + 3] * -s0) << 16));
                }
            } else if (keep) {
#pragma unroll
                for (int k = 0; k < kE; k += 4)
                    *reinterpret_cast<float4*>(po + 4 * j16 + 16 * k) =
                        make_float4(o[k] * s0, o[k + 1] * -s0, o[k + 2] * s0, o[k + 3] * -s0);
                if (i == 0) *pm2 = make_float2(M, L);
            }
        }
        // the next piece's setup writes its decode tables over the merge spaces
        if constexpr (PAGED) __syncthreads();
    };  // item

    if constexpr (PAGED) {
        // Every kv head has the same work (the units' passes over their kv
        // lengths), split into Gh = G / H segments; workgroup b takes head
        // b / Gh and segment seg(b % Gh) of it.  Gh is a multiple of 8 and
        // workgroup b runs on XCD b % 8, so the H workgroups of one segment
        // share an XCD and walk the same tokens at the same time: the heads
        // of a token share its cache lines (cell tib * H + h), and the second
        // reader finds them in that XCD's L2.  The segments of one XCD are
        // consecutive, so the units of a sequence mostly share it too.
        const int Gh = (int)gridDim.x / g.H;
        const int hh = (int)blockIdx.x / Gh;
        const int bl = (int)blockIdx.x - hh * Gh;
        __shared__ UnitRec s_units[kPlanGroups + 1];
        __shared__ int s_plan[7], s_unit;
        const bool planned = pr.units != nullptr;  // by paged_plan_kernel
        int nu, seg, b0, b1;
        if (planned) {
            nu = __builtin_amdgcn_readfirstlane(pr.plan[0]);
            const int total = __builtin_amdgcn_readfirstlane(pr.plan[1]);
            seg = (bl & 7) * (Gh >> 3) + (bl >> 3);
            const Segments sg(total, Gh, pr.inv_segments);
            b0 = sg.bound(seg), b1 = sg.bound(seg + 1);
            if (b0 >= b1) return;  // an empty segment (less work than workgroups)
            // The unit holding work position b0: exactly one u has start(u) <= b0
            // < start(u + 1), or b0 lies before the first unit's first pass
            // (unit 0).
            for (int u = threadIdx.x; u < nu; u += 64 * kWaves)
                if ((u == 0 || pr.units[u].start <= b0) && b0 < pr.units[u + 1].start) s_unit = u;
            __syncthreads();
        } else {
            plan_step(pr, num_queries, num_kv_tokens, Gh, bl, blockIdx.x == 0,
                      reinterpret_cast<int*>(lut), s_units, s_plan);
            nu = __builtin_amdgcn_readfirstlane(s_plan[0]);
            seg = __builtin_amdgcn_readfirstlane(s_plan[3]);
            b0 = __builtin_amdgcn_readfirstlane(s_plan[4]);
            b1 = __builtin_amdgcn_readfirstlane(s_plan[5]);
            if (b0 >= b1) return;
        }
        // (a pass per segment: weight 1)
        const bool ones = !planned && s_plan[1] == s_plan[2];
        const int u_first = __builtin_amdgcn_readfirstlane(planned ? s_unit : s_plan[6]);
        // The walk over the units overlapping the segment, in work order.  Its
        // position lives in LDS (one copy per wave, volatile accesses), so no
        // walk state is held in registers across an item.  The pointer is an
        // LDS one: a generic (flat) access would also wait for the previous
        // piece's partial stores.
        __shared__ int s_walk[kWaves];
        typedef __attribute__((address_space(3))) int lds_int;
        const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        volatile lds_int* walk = (volatile lds_int*)&s_walk[wv];
        if ((threadIdx.x & 63) == 0) walk[0] = u_first;
        for (;;) {
            const int u = __builtin_amdgcn_readfirstlane(walk[0]);
            if (u >= nu) break;
            int first, npos, kv_end, start, useq;
            if (planned) {
                const PagedUnit un = pr.units[u];
                first = un.first, npos = un.npos, kv_end = un.kv_end, start = un.start, useq = un.seq_kv;
            } else {
                const UnitRec un = s_units[u];
                first = __builtin_amdgcn_readfirstlane((int)un.first);
                npos = __builtin_amdgcn_readfirstlane((int)un.npos);
                kv_end = __builtin_amdgcn_readfirstlane(un.kv_end);
                start = __builtin_amdgcn_readfirstlane(un.start);
                useq = __builtin_amdgcn_readfirstlane(un.seq);
            }
            if (start >= b1) break;
            if ((threadIdx.x & 63) == 0) walk[0] = u + 1;
            int x0, x1;
            item_passes(start, (kv_end + kPass - 1) / kPass, ones ? 1 : pass_weight(npos), b0, b1,
                        x0, x1);
            if (x0 < x1) {
                int tid = threadIdx.x;
                asm volatile("" : "+v"(tid));  // opaque per item (see item)
                // partial slot: (unit + segment) * H + head, unique (the
                // pieces of one head form a staircase in (unit, segment))
                item(tid, hh, first, npos, useq, x0 * kPass, min(x1 * kPass, kv_end),
                     (size_t)(u + seg) * g.H + hh);
            }
        }
    } else {
        // Grid (split, kv head, unit), or one dimension of splits x heads x
        // units when there are more units than a grid dimension holds.
        const int groups = (num_queries + kRows - 1) / kRows;
        int split, h, un;
        if (gridDim.x == (unsigned)num_splits) {
            split = blockIdx.x;
            h = blockIdx.y;
            un = blockIdx.z;
        } else {
            split = blockIdx.x % num_splits;
            const int hr = blockIdx.x / num_splits;
            h = hr % g.H;
            un = hr / g.H;
        }
        const int t_begin = split * tokens_per_split;
        item(threadIdx.x, h, un * kNP, min(kNP, groups - un * kNP), 0, t_begin,
             min(t_begin + tokens_per_split, num_kv_tokens), (size_t)split);
    }
}
}  // namespace unit
// Sum of the split partials of one output row (q, h): o = sum_s 2^(m_s - M)
// o_s / sum_s 2^(m_s - M) l_s.  Block = (row, 32-element slice of d), 256
// threads = 8 groups x 32 d.  Group g takes splits g, g + 8, ...: it loads up
// to 16 partials' (m, l, o[d]) in one round, merges them with a running
// maximum, and the 8 groups are merged in LDS.
__global__ __launch_bounds__(256) void attn_mfma_combine_kernel(const float* __restrict__ ws,
                                                                uint16_t* __restrict__ output,
                                                                int H, int num_splits) {
    using namespace mfma;
    constexpr int kBatch = 16;
    __shared__ float red_m[8], red_l[8];
    __shared__ float red_o[8][33];
    // Grid (slice, kv head, query), or one dimension of 4 x rows when there
    // are more queries than a grid dimension holds; row = q * H + h.
    int dq, h, q;
    if (gridDim.x == 4) {
        dq = blockIdx.x;
        h = blockIdx.y;
        q = blockIdx.z;
    } else {
        dq = blockIdx.x & 3;
        const int rw = blockIdx.x >> 2;
        q = rw / H;
        h = rw - q * H;
    }
    const int row = q * H + h;
    const int rg = q / kRows, r = q % kRows;
    const int t = threadIdx.x, dd = t & 31, sg = t >> 5;
    const int d = 32 * dq + dd;
    const size_t base_bid = (size_t)(rg * H + h) * num_splits;
    auto part = [&](int s) { return ws + ((base_bid + s) * kRows + r) * kPartStride; };
    const int S = num_splits;

    float M = kInitMax, L = 0.f, acc = 0.f;
    for (int base = sg; base < S; base += 8 * kBatch) {
        float pm[kBatch], pl[kBatch], po[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
            const int s = base + 8 * k;
            const float* p = part(s < S ? s : base);
            const float2 ml2 = *reinterpret_cast<const float2*>(p + 128);  // (m, l)
            pm[k] = s < S ? ml2.x : kInitMax;
            pl[k] = ml2.y;
            po[k] = p[d];
        }
        float mb = M;
#pragma unroll
        for (int k = 0; k < kBatch; ++k) mb = fmaxf(mb, pm[k]);
        // v_exp_f32 without denormal handling: arguments are <= 0 and a weight
        // below 2^-126 of the largest is negligible.
        const float sc = __builtin_amdgcn_exp2f(M - mb);
        L *= sc;
        acc *= sc;
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
            const float wt = __builtin_amdgcn_exp2f(pm[k] - mb);
            L += pl[k] * wt;
            acc += po[k] * wt;
        }
        M = mb;
    }
    if (dd == 0) {
        red_m[sg] = M;
        red_l[sg] = L;
    }
    red_o[sg][dd] = acc;
    __syncthreads();
    if (t < 32) {
        float Mx = red_m[0];
#pragma unroll
        for (int u = 1; u < 8; ++u) Mx = fmaxf(Mx, red_m[u]);
        float Lt = 0.f, o = 0.f;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const float wt = __builtin_amdgcn_exp2f(red_m[u] - Mx);
            Lt += red_l[u] * wt;
            o += red_o[u][t] * wt;
        }
        output[(size_t)row * 128 + 32 * dq + t] = f2h(Lt > 0.f ? o / Lt : o);
    }
}

// The same merge for few splits: one block per (row group, kv head) item,
// thread t takes row t / 32 and elements 4(t % 32) .. +3 over every split
// (8 in flight).  One block per item instead of 4 per row: for the many short
// items of a batched decode step the block count, not the bytes, is the cost.
constexpr int kItemCombineMaxSplits = 32;
__global__ __launch_bounds__(256) void attn_mfma_combine_items_kernel(
    const float* __restrict__ ws, uint16_t* __restrict__ output, int H, int num_splits,
    int num_queries) {
    using namespace mfma;
    const int item = blockIdx.x;  // h + H * rg
    const int h = item % H, rg = item / H;
    const int t = threadIdx.x, r = t >> 5, d0 = 4 * (t & 31);
    const int S = num_splits;
    const float* base = ws + ((size_t)item * num_splits * kRows + r) * kPartStride;
    float M = kInitMax, L = 0.f;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int b = 0; b < S; b += 8) {
        float pm[8], pl[8];
        float4 po[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const bool ok = b + k < S;
            const float* p = base + (size_t)min(b + k, S - 1) * kRows * kPartStride;
            pm[k] = ok ? p[128] : kInitMax;
            pl[k] = ok ? p[129] : 0.f;
            po[k] = ok ? *reinterpret_cast<const float4*>(p + d0) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        float mb = M;
#pragma unroll
        for (int k = 0; k < 8; ++k) mb = fmaxf(mb, pm[k]);
        const float sc = __builtin_amdgcn_exp2f(M - mb);  // (argument <= 0)
        L *= sc;
        acc.x *= sc;
        acc.y *= sc;
        acc.z *= sc;
        acc.w *= sc;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float wt = __builtin_amdgcn_exp2f(pm[k] - mb);
            L += pl[k] * wt;
            acc.x += po[k].x * wt;
            acc.y += po[k].y * wt;
            acc.z += po[k].z * wt;
            acc.w += po[k].w * wt;
        }
        M = mb;
    }
    const int q = rg * kRows + r;
    if (q >= num_queries) return;
    const auto fin = [&](float o) { return (uint32_t)f2h(L > 0.f ? o / L : o); };
    *reinterpret_cast<uint2*>(output + ((size_t)q * H + h) * 128 + d0) =
        make_uint2(fin(acc.x) | (fin(acc.y) << 16), fin(acc.z) | (fin(acc.w) << 16));
}

// Merge of a paged step's partials.  A row group is position p of unit u; its
// item's passes were cut at segment bounds into pieces, one partial per
// segment they start in (slot unit + segment, position p), and a piece
// starting at or past the group's longest row wrote none.  One wave per (row,
// slice of 4 LS elements): 64 / LS lane groups take the segments in turn, kB
// at a time (every load of a batch in flight together), merge them with a
// running maximum, then the groups are merged across lanes.  LS = 8 (one
// 128-byte line, 8 groups) for few rows, whose unit may lie in a hundred
// segments; LS = D / 4 (a whole row) for many, which have a few each.  Bound by
// its chain of dependent loads: 3 row groups x 4 heads 8.4 -> 4.2 us, 160 x 2
// 6.5 -> 5.3 us, against a block of 256 threads per item that read eight
// segments at a time.
template <int D, int LS>
__global__ __launch_bounds__(64) void attn_paged_combine_kernel(
    const float* __restrict__ ws, uint16_t* __restrict__ output, int H, int num_queries,
    mfma::PagedRows pr) {
    using namespace mfma;
    constexpr int kG = 64 / LS, kSlices = D / (4 * LS), kB = 4;
    const int t = threadIdx.x, grp = t / LS;
    const int d0 = 4 * LS * (blockIdx.x % kSlices) + 4 * (t % LS);
    const int row = blockIdx.x / kSlices;  // ((row group) * H + head) * 8 + row
    const int r = row % kRows, item = row / kRows, h = item % H, rg = item / H;
    const int q = rg * kRows + r;
    if (q >= num_queries) return;
    const PagedUnit un = pr.group_unit[rg];
    const int total = pr.plan[1], G = pr.plan[2];
    const int p = rg - un.first, kv = un.seq_kv, S = un.start;
    // Segment gs holds the item's passes [first(bound(gs)), first(bound(gs + 1))).
    const auto first = [&](int b) { return min(un.n, passes_of(max(b - S, 0), un.w)); };
    int g_lo = 0, g_hi = -1;
    const Segments sg(max(total, 1), G, pr.inv_segments);
    if (un.n > 0 && kv > 0) {
        g_lo = sg.of(S, total);
        g_hi = sg.of(S + un.w * (un.n - 1), total);
    }
    const float* base = ws + ((((size_t)un.index * H + h) * unit::kNP + p) * kRows + r) *
                                 unit::part_stride(D);
    const size_t seg_stride = (size_t)H * unit::kNP * kRows * unit::part_stride(D);
    float M = kInitMax, L = 0.f;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int b = g_lo + grp; b <= g_hi; b += kG * kB) {
        float4 po[kB];
        float2 mlr[kB];
        int okv[kB];
        // (slot gs <= g_hi is one of the item's pieces: the loads are
        // unconditional and all in flight together; the pieces that wrote
        // nothing are dropped after, by a per-lane select rather than a branch
        // whose join would wait for each load in turn)
#pragma unroll
        for (int k = 0; k < kB; ++k) {
            const int gs = min(b + kG * k, g_hi);
            const float* pp = base + seg_stride * gs;
            mlr[k] = *reinterpret_cast<const float2*>(pp + D);
            po[k] = *reinterpret_cast<const float4*>(pp + d0);
            const int x0 = first(sg.bound(gs));
            okv[k] = b + kG * k <= g_hi && x0 < first(sg.bound(gs + 1)) && x0 * unit::kPass < kv;
        }
        __builtin_amdgcn_sched_barrier(0);
        float pm[kB], pl[kB];
#pragma unroll
        for (int k = 0; k < kB; ++k) {
            int ok = okv[k];
            asm volatile("" : "+v"(ok));
            pm[k] = ok ? mlr[k].x : kInitMax;
            pl[k] = ok ? mlr[k].y : 0.f;
            if (!ok) po[k] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
        float mb = M;
#pragma unroll
        for (int k = 0; k < kB; ++k) mb = fmaxf(mb, pm[k]);
        const float sc = __builtin_amdgcn_exp2f(M - mb);  // (argument <= 0)
        L *= sc;
        acc.x *= sc;
        acc.y *= sc;
        acc.z *= sc;
        acc.w *= sc;
#pragma unroll
        for (int k = 0; k < kB; ++k) {
            const float wt = __builtin_amdgcn_exp2f(pm[k] - mb);
            L += pl[k] * wt;
            acc.x += po[k].x * wt;
            acc.y += po[k].y * wt;
            acc.z += po[k].z * wt;
            acc.w += po[k].w * wt;
        }
        M = mb;
    }
    // The lane groups (lanes LS apart), pairwise.
    const auto merge = [&](auto lanes) {
        constexpr int X = decltype(lanes)::value;
        if constexpr (X >= LS) {
            const float Mp = lane_xor<X>(M), mn = fmaxf(M, Mp);
            const float a = __builtin_amdgcn_exp2f(M - mn), c = __builtin_amdgcn_exp2f(Mp - mn);
            L = L * a + lane_xor<X>(L) * c;
            acc.x = acc.x * a + lane_xor<X>(acc.x) * c;
            acc.y = acc.y * a + lane_xor<X>(acc.y) * c;
            acc.z = acc.z * a + lane_xor<X>(acc.z) * c;
            acc.w = acc.w * a + lane_xor<X>(acc.w) * c;
            M = mn;
        }
    };
    merge(std::integral_constant<int, 8>{});
    merge(std::integral_constant<int, 16>{});
    merge(std::integral_constant<int, 32>{});
    if (t >= LS) return;
    const auto fin = [&](float o) { return (uint32_t)f2h(L > 0.f ? o / L : o); };
    store_h4(output + ((size_t)q * H + h) * D + d0, fin(acc.x) | (fin(acc.y) << 16),
             fin(acc.z) | (fin(acc.w) << 16));
}

// Inclusive scan over the 1024 threads of a block (16 waves) with an
// associative op: within each wave by shuffles, then over the wave totals.
template <typename Op>
__device__ int block_scan_1024(int v, int ident, int* s_tot, Op op) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(v, d);
        if (lane >= d) v = op(v, o);
    }
    if (lane == 63) s_tot[wv] = v;
    __syncthreads();
    // The earlier waves' totals: all 16 read at once (one LDS round trip),
    // then combined below this wave's index.
    int tot[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) tot[k] = s_tot[k];
    int pre = ident;
#pragma unroll
    for (int k = 0; k < 16; ++k)
        if (k < wv) pre = op(pre, tot[k]);
    __syncthreads();  // s_tot is reused by the next scan
    return op(pre, v);
}

// The plan of a paged step of more than unit::kPlanGroups row groups, one
// block of 1024 threads.  Row groups (8 rows
// of one sequence) form units: each run of consecutive groups of one
// sequence is cut into units of U groups from its start, the last one
// shorter.  A unit's items (one per kv head) are n = ceil(kv_end / pass)
// passes over its longest row (at most max_kv_len), a pass weighing w: with
// U = 4, 4 for a unit of more than two positions (the two-tile loop) and 3
// otherwise, about their measured cost ratio.  Work positions are given out
// in unit order; a unit with passes first takes kPieceCost positions that no
// pass occupies (its start is its first pass): a workgroup pays a piece's
// setup (query rotation, decode tables, a first chunk with nothing in flight)
// for every unit it starts, so a segment holding unit starts gets less pass
// work.  The groups are taken 1024 at a time, carrying the run start, the
// unit count and the work total from window to window.
template <int U>
__global__ __launch_bounds__(1024) void paged_plan_kernel(
    const int32_t* __restrict__ row_seq, const int32_t* __restrict__ row_kv_len, int num_rows,
    int groups, int pass, int max_kv_len, int segments, mfma::PagedUnit* __restrict__ units,
    mfma::PagedUnit* __restrict__ group_unit, int32_t* __restrict__ plan) {
    static_assert(U >= 1 && U <= 4 && (U & (U - 1)) == 0, "1, 2 or 4 groups per unit");
    using mfma::kRows;
    constexpr int kWin = 1024;
    __shared__ int s_sq[kWin + U], s_gk[kWin + U], s_tot[16], s_carry[4];
    const int j = threadIdx.x;
    // The group's longest row (rows past num_rows: 0).  The loads are
    // unconditional (a row past the end re-reads the last row), so the eight
    // go out together: a load under a condition sits in a branch whose join
    // waits for it, one memory latency per row.
    auto load_kv = [&](int gi, int (&v)[kRows]) {
#pragma unroll
        for (int k = 0; k < kRows; ++k) v[k] = row_kv_len[min(gi * kRows + k, num_rows - 1)];
    };
    auto group_kv = [&](int gi, const int (&v)[kRows]) {
        int m = 0;
#pragma unroll
        for (int k = 0; k < kRows; ++k)
            if (gi * kRows + k < num_rows) m = max(m, v[k]);
        return min(m, max_kv_len);
    };
    const auto add = [](int a, int b) { return a + b; };
    const auto mx = [](int a, int b) { return max(a, b); };
    int c_units = 0, c_work = 0, c_rs = 0, c_sq = 0;
    for (int base = 0; base < groups; base += kWin) {
        const int gi = base + j;
        const bool in = gi < groups;
        // (groups past the end load the last group, unconditionally, then drop it)
        const int gc = min(gi, groups - 1);
        const int gx = min(base + kWin + j, groups - 1);  // look-ahead (threads j < U - 1)
        int kvr[kRows], kvx[kRows];
        const int sq_raw = row_seq[(size_t)gc * kRows];
        const int sqx_raw = row_seq[(size_t)gx * kRows];
        load_kv(gc, kvr);
        load_kv(gx, kvx);
        __builtin_amdgcn_sched_barrier(0);  // all 18 loads in flight before any is used
        const int gk_raw = group_kv(gc, kvr);
        const int gkx_raw = group_kv(gx, kvx);
        const int sq = in ? sq_raw : 0;
        s_sq[j] = sq;
        s_gk[j] = in ? gk_raw : 0;
        {  // look-ahead for units that straddle the window's end: threads j < U - 1
            // write slot kWin + j, the others the spare last slot (never read),
            // so no branch holds the look-ahead loads back
            const bool inx = j < U - 1 && base + kWin + j < groups;
            s_sq[kWin + min(j, U - 1)] = inx ? sqx_raw : 0;
            s_gk[kWin + min(j, U - 1)] = inx ? gkx_raw : 0;
        }
        __syncthreads();
        const int prev = j > 0 ? s_sq[j - 1] : c_sq;
        const bool new_run = in && (gi == 0 || sq != prev);
        int rs = block_scan_1024(new_run ? gi : -1, -1, s_tot, mx);
        if (rs < 0) rs = c_rs;
        const bool start = in && ((gi - rs) & (U - 1)) == 0;
        int c = 1, kv = s_gk[j];
#pragma unroll
        for (int k = 1; k < U; ++k)
            if (c == k && gi + k < groups && s_sq[j + k] == sq) {
                ++c;
                kv = max(kv, s_gk[j + k]);
            }
        const int w = U > 2 ? unit::pass_weight(c) : 1;
        const int n = (kv + pass - 1) / pass;
        const int lead = n > 0 ? unit::kPieceCost : 0;
        const int work = start ? lead + w * n : 0;  // per kv head (every head has it)
        const int ui = block_scan_1024(start ? 1 : 0, 0, s_tot, add);
        const int wi = block_scan_1024(work, 0, s_tot, add);
        if (start) {
            const int o = c_units + ui - 1;
            const mfma::PagedUnit rec{gi, c, kv, c_work + wi - work + lead, n, w, o, sq};
            units[o] = rec;
            for (int k = 0; k < c; ++k) {
                mfma::PagedUnit gu = rec;
                gu.seq_kv = s_gk[j + k];
                group_unit[gi + k] = gu;
            }
        }
        if (j == kWin - 1) {  // window totals (inclusive scans at the last thread)
            s_carry[0] = ui;
            s_carry[1] = wi;
            s_carry[2] = rs;
            s_carry[3] = s_sq[min(groups - base, kWin) - 1];
        }
        __syncthreads();
        c_units += s_carry[0];
        c_work += s_carry[1];
        c_rs = s_carry[2];
        c_sq = s_carry[3];
        __syncthreads();  // before the next window rewrites s_sq and s_carry
    }
    if (j == 0) {
        units[c_units] = mfma::PagedUnit{0, 0, 0, c_work, 0, 1, c_units, 0};  // sentinel
        plan[0] = c_units;
        plan[1] = c_work;
        plan[2] = segments;
    }
}

// ===========================================================================
// Decode over slot-mapped tokens: the reference's fused attention entries
// (src/cuda/tq_turbo_prod_kernels.cu:439-571, 650-671;
// src/cuda/tq_turbo_mse_kernels.cu:302-417, 459-479) for D = 64, 128 and
// turbo_prod / turbo_mse pages.
//
// Flash-decoding split-K on a (split, kv head, row group) grid, 8 waves of
// 32-token chunks per workgroup (QK: A = decoded K, B = the rotated query as
// fp16 hi/lo columns; PV: A = P', B = decoded V), with a setup and a chunk
// loop cut to what the decode needs:
//  - one LDS lookup per K code byte returns two fp16 pairs: turbo_prod's
//    aK*K3 pair and its pair of residual signs (+-1; no VALU builds the sign
//    matrix), turbo_mse's hi and lo parts of aV*V4 (its V lookups read the
//    hi pair of the same entry);
//  - the tables are built in registers from compile-time constants while the
//    slots and codes are in flight (no staging pass);
//  - each wave rotates one query row and stores its fp16 hi and lo parts
//    straight into the B-operand layout: one barrier for the whole setup;
//  - P' = p * vs / aV enters the PV product as its fp16 hi part, or on the
//    lo columns as fp16(p * vs / aV - hi) of the exact product (three
//    mixed-precision ops per value pair and lane);
//  - per split and row the partial o[128] and (m, l) go to two arrays, the
//    (m, l) of one row contiguous over the splits, for
//    attn_decode_combine_kernel.
// ===========================================================================
namespace dec {
using namespace mfma;

// LDS layout of the tables (entries as decode_table_words describes) (32 copies of each entry, copy c at 4c; lane l
// reads copy l % 32, so a half-wave's random lookups hit distinct banks):
//   S table: byte 256b + 4c;
//   K table: byte kOffK + 256b + 4c (turbo_mse's V lookups read it too);
//   turbo_prod's V table: kOffK + 256b + 128 + 4c;
//   turbo_prod's V lo table (head_dim 64): 256b + 128 + 4c, c < kLoCopies (the
//   S rows' upper halves; the last four copies of the last row would lie past
//   kOffK, so lanes 28 .. 31 of a half-wave read copies 0 .. 3).
// A K lookup reads its S and K entries from one address register with
// offsets 0 and kOffK: no two-address LDS read reaches that pair (ds_read2
// spans up to 1020 bytes, ds_read2st64 multiples of 256), so each result
// goes straight into its MFMA operand registers.
constexpr int kOffK = 65520;
constexpr int kLutWords = (kOffK + 256 * 256) / 4;
constexpr int kLoCopies = 28;
static_assert(256 * 255 + 128 + 4 * kLoCopies <= kOffK, "the V lo rows end below the K table");

// LDS address of copy (lane & 31) of entry `byte b of word` in a table of
// 256-byte entries at `base` (base = table + copy offset): v_perm puts the
// code byte in byte 1, and byte 1 of the base is added back.
__device__ __forceinline__ uint32_t lut_addr(uint32_t word, int b, uint32_t base) {
    return __builtin_amdgcn_perm(word, base, 0x03020000u | ((4u + b) << 8)) + (base & 0xFF00u);
}

// fp16 pair of x0 = a0 * b0, x1 = a1 * b1 for this lane's MFMA column: the
// hi parts fp16(x), or with lomask = ~0 the lo parts fp16(x - hi) of the
// exact products (v_fma_mix: one rounding to fp16).
__device__ __forceinline__ uint32_t hilo_pair(float a0, float b0, float a1, float b1,
                                              uint32_t lomask) {
    uint32_t h, r;
    asm("v_fma_mixlo_f16 %0, %1, %2, 0 op_sel_hi:[0,0,0]\n\t"
        "v_fma_mixhi_f16 %0, %3, %4, 0 op_sel_hi:[0,0,0]"
        : "=&v"(h)
        : "v"(a0), "v"(b0), "v"(a1), "v"(b1));
    const uint32_t m = h & lomask;
    asm("v_fma_mixlo_f16 %0, %1, %2, -%5 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %0, %3, %4, -%5 op_sel:[0,0,1] op_sel_hi:[0,0,1]"
        : "=&v"(r)
        : "v"(a0), "v"(b0), "v"(a1), "v"(b1), "v"(m));
    return r;
}

constexpr int kWaves = 8, kChunk = 32, kPass = kWaves * kChunk;
// Partial of (split, row): o[D] at po[(pid * 8 + r) * D], (m, l) at
// pml[(item * 8 + r) * S + split] with pid = item * S + split and item =
// row group * H + kv head.
constexpr size_t part_bytes(int D) { return kRows * (D + 2) * sizeof(float); }

// D = 128, or D = 64: half the dims per token (two QK k-steps instead of
// four, four PV tiles instead of eight), 8-byte K and 2-byte V loads per
// lane.  D = 64 also carries what keeps it as exact as fp32 arithmetic: the
// fp16 lo parts of V (a second PV product in its own accumulators; the
// table's hi parts alone are 5e-5 off in the mean, a quarter of the output's
// own fp16 rounding) and of turbo_prod's K (in the S table, a third QK
// product; the signs are built in registers: logits of magnitude 60, outlier
// channels shared by q and k, are 6e-4 off without it), and powers of two, one
// per query row and one per wave for V, that hold their fp16 parts in range
// whatever their magnitudes.  Bound by its dependent loads and
// the setup, as D = 128: 7 rows x 2 heads x 6,001 tokens (turbo_mse) take 6.0
// (split) + 2.9 us (combine); the generic one-wave-per-row kernels, whose
// cross-lane sum per token and serial merge over 147 splits this replaces,
// took 22.7 + 70.2 us.
template <int SCH, int D>
__global__ __launch_bounds__(64 * kWaves) void attn_decode_split_kernel(
    const uint16_t* __restrict__ query, const uint8_t* __restrict__ pool,
    const int32_t* __restrict__ slots, float* __restrict__ po, float2* __restrict__ pml,
    uint16_t* __restrict__ output, float inv, int num_queries, int num_kv_tokens,
    int tokens_per_split, int num_splits, PageGeom g) {
    constexpr bool PROD = SCH == kSchProd;
    static_assert(SCH == kSchProd || SCH == kSchMse, "turbo_prod or turbo_mse pages");
    static_assert(D == 128 || D == 64, "head_dim 64 or 128");
    constexpr int kS = D / 32;       // QK k-steps; lane group gq holds dims [D/4 gq, D/4 gq + D/4)
    constexpr int kNT = D / 16;      // PV tiles: lane i holds dims kNT i .. + kNT - 1
    constexpr int kL = D / 2;        // lanes of a row held two values per lane
    constexpr bool VLO = D == 64, QSCALE = D == 64, KLO = D == 64 && PROD, VSCALE = D == 64;
    // The decode tables (layout above); after the chunk loop the space holds
    // the waves' results for the merge.
    __shared__ __attribute__((aligned(256))) uint32_t lut[kLutWords];
    __shared__ uint4 bqs[kS][64];  // QK B operand of k-step s for lane l
    __shared__ uint64_t tko[kWaves][kChunk], tvo[kWaves][kChunk];
    __shared__ float4 tsc[kWaves][kChunk];  // per token: K scale, residual scale, vs / aV, bias
    __shared__ float mm[kWaves][kRows], ml[kWaves][kRows];
    __shared__ float rsc[kRows];  // QSCALE: the rows' power of two
    float(*mo)[kRows][D] = reinterpret_cast<float(*)[kRows][D]>(&lut[0]);
    static_assert(sizeof(float) * kWaves * kRows * D <= sizeof(lut), "merge space");

    int split, h, rg;
    if (gridDim.x == (unsigned)num_splits) {
        split = blockIdx.x;
        h = blockIdx.y;
        rg = blockIdx.z;
    } else {  // one dimension of splits x heads x row groups
        split = blockIdx.x % num_splits;
        const int hr = blockIdx.x / num_splits;
        h = hr % g.H;
        rg = hr / g.H;
    }
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 15, gq = lane >> 4;
    const int jl = lane & (kL - 1);  // this lane's pair of a row (D = 64: lanes l and l + 32 alike)
    const int t_begin = split * tokens_per_split;
    const int t_end = min(num_kv_tokens, t_begin + tokens_per_split);
    // logit scale per unit ks (log2(e) / alpha folded at compile time: no run-time division)
    const float ck = inv * (PROD ? kLog2e / kAlphaK : kLog2e / kAlphaV);
    const float cr = inv * kLog2e;                                 // residual: ks * re
    constexpr float iav = 1.0f / kAlphaV;

    // 1. Loads, in the order they are needed: this wave's query row, the
    //    first chunk's slots, then the decode-table words.
    const int qrow = rg * kRows + w;
    const uint32_t qraw = *reinterpret_cast<const uint32_t*>(
        query + ((size_t)min(qrow, num_queries - 1) * g.H + h) * D + 2 * jl);
    int t0 = t_begin + w * kChunk;
    auto load_slot = [&](int t) -> int {
        return slots[max(min(t + (lane & (kChunk - 1)), t_end - 1), 0)];
    };
    const int slot0 = load_slot(t0);
    // 2. The chunk's codes and per-token scales.  slot -> cell offsets
    //    (exchanged through this wave's LDS rows) -> scale and code loads.
    //    Tokens past the range or with a negative slot read the first bytes
    //    of the query instead (always valid memory) and get bias -inf.
    struct Chunk {
        uint32_t kw[2][kS];  // K: tile tau, token 16 tau + i, bytes [4 kS gq, 4 kS gq + 4 kS)
        uint32_t vw[8];  // V: k-index 8 gq + e (token below), bytes [D/32 i, D/32 i + D/32)
        uint16_t ks, re, vs;
        bool valid;
    };
    const uint64_t dummy_off =
        (uint64_t)(reinterpret_cast<uintptr_t>(query) - reinterpret_cast<uintptr_t>(pool));
    auto fetch = [&](int tc, int slot, Chunk& c) {
        c.valid = tc + (lane & (kChunk - 1)) < t_end && slot >= 0;
        int page, tib;
        split_slot(c.valid ? slot : 0, g, page, tib);
        const uint64_t cell = (uint64_t)(tib * g.H + h);
        const uint64_t pb = (uint64_t)page * g.page_size;
        const uint64_t so = pb + cell * g.scale_stride;
        c.ks = ld_u16_nt(pool + (c.valid ? so + g.ks_off : dummy_off));
        c.vs = ld_u16_nt(pool + (c.valid ? so + g.vs_off : dummy_off + 2));
        c.re = PROD ? ld_u16_nt(pool + (c.valid ? so + g.kres_off : dummy_off + 4)) : (uint16_t)0;
        tko[w][lane & (kChunk - 1)] = c.valid ? pb + g.kc_off + cell * g.code_stride : dummy_off;
        tvo[w][lane & (kChunk - 1)] = c.valid ? pb + g.vc_off + cell * g.code_stride : dummy_off;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int tau = 0; tau < 2; ++tau) {
            const uint8_t* kp = pool + (tko[w][16 * tau + i] + 4 * kS * gq);
            if constexpr (D == 128) {
                const uint4 x = ld_u4_nt(kp);
                c.kw[tau][0] = x.x, c.kw[tau][1] = x.y, c.kw[tau][2] = x.z, c.kw[tau][3] = x.w;
            } else {
                const uint2 x = ld_u2_nt(kp);
                c.kw[tau][0] = x.x, c.kw[tau][1] = x.y;
            }
        }
        // k-index 8 gq + e is token 4 gq + e (e < 4) or 16 + 4 gq + (e - 4)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int tok = e < 4 ? 4 * gq + e : 16 + 4 * gq + (e - 4);
            const uint8_t* vp = pool + (tvo[w][tok] + D / 32 * i);
            c.vw[e] = D == 128 ? ld_u32_nt(vp) : (uint32_t)ld_u16_nt(vp);
        }
    };
    Chunk cur;
    fetch(t0, slot0, cur);
    int slot_nx = load_slot(t0 + kPass);
    __builtin_amdgcn_sched_barrier(0);  // the code loads go out before any setup work

    // The tables' words, computed in registers while the codes are in flight
    // (no memory traffic; each 16-byte store writes four copies).
    const TableWords<PROD> tw = decode_table_words<PROD, KLO>(w, lane);
    uint32_t vlo[4];
    if constexpr (VLO && PROD) lo_table_words(w, lane, vlo);
    // 3. This wave's query row: qrot = WHT(q * s) * inv, stored as fp16 hi
    //    and lo parts into the B operand (column 2w: hi, 2w + 1: lo; lane l
    //    holds d = 2l, 2l + 1: k-group l / (4 kS), k-step (l / 4) % kS, halves
    //    2(l % 4), + 1 of the half8).
    {
        const float sh = (h & 1) ? -1.0f : 1.0f;
        float q0 = h2f(qraw & 0xffff) * sh, q1 = h2f(qraw >> 16) * (-sh);
        wht_pair<kL>(q0, q1, lane);
        const bool live = qrow < num_queries;
        q0 = live ? q0 * inv : 0.0f;
        q1 = live ? q1 * inv : 0.0f;
        if constexpr (QSCALE) {
            // the row's largest |q| scaled into [0.5, 1) (a zero or non-finite
            // row is left as it is); its logits are multiplied back
            const int ex = scale_exp(max_lanes<kL>(fmaxf(fabsf(q0), fabsf(q1))));
            q0 = __builtin_amdgcn_ldexpf(q0, -ex);
            q1 = __builtin_amdgcn_ldexpf(q1, -ex);
            if (lane == 0) rsc[w] = __builtin_amdgcn_ldexpf(1.0f, ex);
        }
        const uint32_t hi = pack_h2(q0, q1);
        const uint32_t lo = lo_pair(q0, q1, hi);
        uint32_t* b = reinterpret_cast<uint32_t*>(
            &bqs[(jl >> 2) & (kS - 1)][16 * (jl / (4 * kS)) + 2 * w]);
        b[jl & 3] = hi;  // (D = 64: both halves of the wave write the same words)
        b[4 + (jl & 3)] = lo;  // the next lane's (column 2w + 1) half8
    }
    // 4. The decode tables.
    store_decode_tables<PROD>(lut, kOffK / 4, w, lane, tw);
    if constexpr (VLO && PROD) {
        if ((lane & 7) < kLoCopies / 4) {
#pragma unroll
            for (int k = 0; k < 4; ++k)
                *reinterpret_cast<u32x4*>(
                    &lut[(32 * w + 8 * k + (lane >> 3)) * 64 + 32 + 4 * (lane & 7)]) =
                    (u32x4){vlo[k], vlo[k], vlo[k], vlo[k]};
        }
    }
    lds_barrier();
    half8 bq[kS];
#pragma unroll
    for (int s = 0; s < kS; ++s) bq[s] = __builtin_bit_cast(half8, bqs[s][lane]);

    // Lookup bases: copy lane % 32 of entry 0 of the S table (the K table
    // is kOffK above it; turbo_mse's V lookups read it that way), and of
    // turbo_prod's V table.
    const uint32_t basek = (uint32_t)reinterpret_cast<uintptr_t>((lds_u32*)&lut[lane & 31]);
    const uint32_t basev =
        PROD ? (uint32_t)reinterpret_cast<uintptr_t>((lds_u32*)&lut[kOffK / 4 + 32 + (lane & 31)])
             : basek;
    constexpr uint32_t offv = PROD ? 0u : (uint32_t)kOffK;
    // VLO: base of the V lo lookups, whose hi pair is kOffK above (turbo_prod:
    // its copies of the S rows' upper halves; turbo_mse: the S table)
    const uint32_t basel =
        PROD ? (uint32_t)reinterpret_cast<uintptr_t>(
                   (lds_u32*)&lut[32 + ((lane & 31) < kLoCopies ? lane & 31 : (lane & 31) - kLoCopies)])
             : basek;
    const float qsc = QSCALE ? ck * rsc[i >> 1] : 1.0f;
    const bool lo_col = (i & 1) != 0;
    const uint32_t lomask = lo_col ? 0xFFFFFFFFu : 0u;

    float m_run = kInitMax, r_run = kInitMax, l_run = 0.0f;  // maximum, reference, sum
    f32x4 acc[kNT], acl[VLO ? kNT : 1];  // PV sums; VLO: of V's lo parts (x 2^kLoShift)
#pragma unroll
    for (int v = 0; v < kNT; ++v) acc[v] = (f32x4){0.f, 0.f, 0.f, 0.f};
    if constexpr (VLO) {
#pragma unroll
        for (int v = 0; v < kNT; ++v) acl[v] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    bool first = true;
    VPower vp;  // VSCALE

    while (t0 < t_end) {  // wave-uniform
        {
            const float ks = h2f(cur.ks), vs = h2f(cur.vs), re = PROD ? h2f(cur.re) : 0.0f;
            const float kx = QSCALE ? 1.0f : ck, kr = QSCALE ? kAlphaK : cr;
            const float4 sc = PROD ? make_float4(ks * kx, ks * re * kr, vs * iav, 0.0f)
                                   : make_float4(ks * kx, QSCALE ? low_factor(ks) : ks * kx * kLoScale,
                                                 vs * iav, 0.0f);
            tsc[w][lane & (kChunk - 1)] = cur.valid ? sc : make_float4(0.f, 0.f, 0.f, -INFINITY);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if constexpr (VSCALE) vp.raise(cur.valid ? cur.vs : 0u);
        Chunk nxt;
        const int t1 = t0 + kPass;
        if (t1 < t_end) {  // codes of the next chunk, slots of the one after
            fetch(t1, slot_nx, nxt);
            slot_nx = load_slot(t1 + kPass);
        }
        // Per-token scales of this lane's logits (read before the lookups:
        // LDS reads complete in order).
        float4 scv[2][4];
#pragma unroll
        for (int tau = 0; tau < 2; ++tau)
#pragma unroll
            for (int e = 0; e < 4; ++e) scv[tau][e] = tsc[w][16 * tau + 4 * gq + e];
        // QK: every K lookup of the chunk issued before the first MFMA.
        half8 ka[2][kS], kb[2][kS];
#pragma unroll
        for (int tau = 0; tau < 2; ++tau) {
#pragma unroll
            for (int s = 0; s < kS; ++s) {
                uint32_t e0[4], e1[4];  // K entries, S entries
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const uint32_t a = lut_addr(cur.kw[tau][s], b, basek);
                    e0[b] = *reinterpret_cast<const lds_u32*>(a + kOffK);
                    e1[b] = *reinterpret_cast<const lds_u32*>(a);
                }
                ka[tau][s] = as_h8(e0[0], e0[1], e0[2], e0[3]);
                kb[tau][s] = as_h8(e1[0], e1[1], e1[2], e1[3]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        f32x4 cb[2], cs[2];
#pragma unroll
        for (int tau = 0; tau < 2; ++tau) {
            cb[tau] = (f32x4){0.f, 0.f, 0.f, 0.f};
            cs[tau] = cb[tau];
#pragma unroll
            for (int s = 0; s < kS; ++s) {
                if constexpr (KLO) {  // (K's lo parts first, see unit::)
                    cb[tau] = mma(kb[tau][s], bq[s], cb[tau]);
                    cs[tau] = mma(sign_octet(cur.kw[tau][s]), bq[s], cs[tau]);
                } else {
                    cb[tau] = mma(ka[tau][s], bq[s], cb[tau]);
                    cs[tau] = mma(kb[tau][s], bq[s], cs[tau]);  // prod: residual signs; mse: lo parts
                }
            }
            if constexpr (KLO)
#pragma unroll
                for (int s = 0; s < kS; ++s) cb[tau] = mma(ka[tau][s], bq[s], cb[tau]);
        }
        // V lookups (B operands of PV), in flight during the softmax.
        uint32_t bv[kNT][4];  // [N-tile v = d - kNT i][token pair]
        uint32_t bl[VLO ? kNT : 1][4];
        if constexpr (D == 128) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t we = cur.vw[2 * q], wo = cur.vw[2 * q + 1];
                const uint32_t lob = (we & 0x0F0F0F0Fu) | ((wo & 0x0F0F0F0Fu) << 4);
                const uint32_t hib = ((we >> 4) & 0x0F0F0F0Fu) | (wo & 0xF0F0F0F0u);
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    bv[2 * b][q] = *reinterpret_cast<const lds_u32*>(lut_addr(lob, b, basev) + offv);
                    bv[2 * b + 1][q] = *reinterpret_cast<const lds_u32*>(lut_addr(hib, b, basev) + offv);
                }
            }
        } else {
            // two token pairs per word (a lane's row part is two bytes)
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const uint32_t we = cur.vw[4 * p] | (cur.vw[4 * p + 2] << 16);
                const uint32_t wo = cur.vw[4 * p + 1] | (cur.vw[4 * p + 3] << 16);
                const uint32_t lob = (we & 0x0F0F0F0Fu) | ((wo & 0x0F0F0F0Fu) << 4);
                const uint32_t hib = ((we >> 4) & 0x0F0F0F0Fu) | (wo & 0xF0F0F0F0u);
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const int v = 2 * (b & 1), q = 2 * p + (b >> 1);
                    const uint32_t a0 = lut_addr(lob, b, basel), a1 = lut_addr(hib, b, basel);
                    bv[v][q] = *reinterpret_cast<const lds_u32*>(a0 + kOffK);
                    bl[v][q] = *reinterpret_cast<const lds_u32*>(a0);
                    bv[v + 1][q] = *reinterpret_cast<const lds_u32*>(a1 + kOffK);
                    bl[v + 1][q] = *reinterpret_cast<const lds_u32*>(a1);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // Logits (base 2; QSCALE: before their row's factor qsc) of tokens
        // 16 tau + 4 gq + e; hi + lo columns summed.
        float lg[2][4];
        float mloc = -INFINITY;
#pragma unroll
        for (int tau = 0; tau < 2; ++tau)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float4 sc = scv[tau][e];
                const float sb = QSCALE ? pair_even(cb[tau][e]) : cb[tau][e] + quad_xor<1>(cb[tau][e]);
                float sr = cs[tau][e] + quad_xor<1>(cs[tau][e]);
                if constexpr (QSCALE && !PROD)
                    sr = fmaf(pair_odd(cb[tau][e]), (float)(1 << kLoShift), sr);
                float low = fmaf(sr, sc.y, sc.w);
                if constexpr (QSCALE && PROD) low = fmaf(pair_odd(cb[tau][e]), sc.x, low);
                lg[tau][e] = fmaf(sb, sc.x, low);
                mloc = fmaxf(mloc, lg[tau][e]);
            }
        mloc = lane_xor_reduce<16>(mloc, [](float x, float y) { return fmaxf(x, y); });
        mloc = lane_xor_reduce<32>(mloc, [](float x, float y) { return fmaxf(x, y); });
        // v_exp_f32 without denormal handling: arguments are <= 0 and a weight
        // below 2^-126 of the running maximum is negligible.
        m_run = fmaxf(m_run, QSCALE ? mloc * qsc : mloc);
        const float ref = VSCALE ? m_run - vp.k : m_run;
        const float alpha = first ? 0.0f : __builtin_amdgcn_exp2f(r_run - ref);
        r_run = ref;
        float lsum = 0.0f;
#pragma unroll
        for (int tau = 0; tau < 2; ++tau)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                lg[tau][e] = __builtin_amdgcn_exp2f(QSCALE ? fmaf(lg[tau][e], qsc, -ref)
                                                           : lg[tau][e] - ref);
                lsum += lg[tau][e];
            }
        l_run = l_run * alpha + lsum;
        if (!first && __any(alpha != 1.0f)) {
            // acc lane (d, g) holds columns 4g .. 4g + 3 = rows 2g, 2g + 1
            const float a0 = __shfl(alpha, 4 * gq), a1 = __shfl(alpha, 4 * gq + 2);
#pragma unroll
            for (int v = 0; v < kNT; ++v) {
                acc[v][0] *= a0;
                acc[v][1] *= a0;
                acc[v][2] *= a1;
                acc[v][3] *= a1;
                if constexpr (VLO) {
                    acl[v][0] *= a0;
                    acl[v][1] *= a0;
                    acl[v][2] *= a1;
                    acl[v][3] *= a1;
                }
            }
        }
        // PV: P' = p * vs / aV as this column's fp16 part; k-index 8 gq + e is
        // the logit of tile e / 4, element e % 4.
        const half8 ap = as_h8(hilo_pair(lg[0][0], scv[0][0].z, lg[0][1], scv[0][1].z, lomask),
                               hilo_pair(lg[0][2], scv[0][2].z, lg[0][3], scv[0][3].z, lomask),
                               hilo_pair(lg[1][0], scv[1][0].z, lg[1][1], scv[1][1].z, lomask),
                               hilo_pair(lg[1][2], scv[1][2].z, lg[1][3], scv[1][3].z, lomask));
#pragma unroll
        for (int v = 0; v < kNT; ++v)
            acc[v] = mma(ap, as_h8(bv[v][0], bv[v][1], bv[v][2], bv[v][3]), acc[v]);
        if constexpr (VLO) {
#pragma unroll
            for (int v = 0; v < kNT; ++v)
                acl[v] = mma(ap, as_h8(bl[v][0], bl[v][1], bl[v][2], bl[v][3]), acl[v]);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        cur = nxt;
        t0 = t1;
        first = false;
    }

    // Wave results: l summed over the 4 lane groups of each column; o rows
    // from the hi + lo columns.  Then the waves are merged per row, the
    // inverse WHT and sign flip applied, and the partial written.
    {
        float l_tot = lane_xor_reduce<16>(l_run, [](float x, float y) { return x + y; });
        l_tot = lane_xor_reduce<32>(l_tot, [](float x, float y) { return x + y; });
        if (gq == 0 && !lo_col) {
            mm[w][i >> 1] = r_run;
            ml[w][i >> 1] = l_tot;
        }
    }
    lds_barrier();  // every wave is done with the tables mo overwrites
#pragma unroll
    for (int v = 0; v < kNT; ++v) {
        float x0 = acc[v][0] + acc[v][1], x1 = acc[v][2] + acc[v][3];
        if constexpr (VLO) {
            x0 = fmaf(acl[v][0] + acl[v][1], kLoScale, x0);
            x1 = fmaf(acl[v][2] + acl[v][3], kLoScale, x1);
        }
        mo[w][2 * gq][kNT * i + v] = x0;
        mo[w][2 * gq + 1][kNT * i + v] = x1;
    }
    lds_barrier();
    const int r = w;  // this wave's row of the group
    if (rg * kRows + r >= num_queries) return;  // wave-uniform, after the last barrier
    float M = mm[0][r];
#pragma unroll
    for (int u = 1; u < kWaves; ++u) M = fmaxf(M, mm[u][r]);
    float L = 0.f, o0 = 0.f, o1 = 0.f;
#pragma unroll
    for (int u = 0; u < kWaves; ++u) {
        const float wt = __builtin_amdgcn_exp2f(mm[u][r] - M);  // (argument <= 0)
        const float2 ov = *reinterpret_cast<const float2*>(&mo[u][r][2 * jl]);
        L += ml[u][r] * wt;
        o0 += ov.x * wt;
        o1 += ov.y * wt;
    }
    wht_pair<kL>(o0, o1, lane);
    const float s0 = (h & 1) ? -inv : inv;
    if (num_splits == 1) {  // nothing to merge: the output itself
        o0 *= s0;
        o1 *= -s0;
        if (D == 128 || lane < kL)
            store_h2(output + ((size_t)(rg * kRows + r) * g.H + h) * D + 2 * jl,
                     (uint32_t)f2h(L > 0.f ? o0 / L : o0) | ((uint32_t)f2h(L > 0.f ? o1 / L : o1) << 16));
        return;
    }
    const size_t item = (size_t)rg * g.H + h;
    const size_t pid = item * num_splits + split;
    if (D == 128 || lane < kL)
        *reinterpret_cast<float2*>(po + (pid * kRows + r) * D + 2 * jl) =
            make_float2(o0 * s0, o1 * -s0);
    if (lane == 0) pml[(item * kRows + r) * num_splits + split] = make_float2(M, L);
}

// Sum of the split partials of one output row (q, h): o = sum_s 2^(m_s - M)
// o_s / sum_s 2^(m_s - M) l_s.  One wave per (row, 8-element slice of d):
// lane = 8 split groups x 8 elements; group j takes splits j, j + 8, ..., kB
// at a time (every load of a batch in flight together), merges them with a
// running maximum, then the groups are merged across lanes (no LDS, no
// barrier).  kB is the smallest of 2, 4 and 16 that takes S splits in one
// batch: loads past S re-read a split, so a batch of 16 at few splits is
// mostly repeats.  The 4 slices of one 128-byte line of the partials run on one
// XCD (block b on XCD b % 8), so three of them find the line in that XCD's
// L2.
template <int D, int kB>
__global__ __launch_bounds__(64) void attn_decode_combine_kernel(
    const float* __restrict__ po, const float2* __restrict__ pml, uint16_t* __restrict__ output,
    int H, int rows, int S) {
    using namespace mfma;
    const int b = blockIdx.x;
    const int xcd = b & 7, m = b >> 3;
    constexpr int kLines = D / 32;     // 128-byte lines of a partial row
    const int p = (m >> 2) * 8 + xcd;  // (row, line) pair
    const int row = p / kLines;
    if (row >= rows) return;
    const int t = threadIdx.x, dd = t & 7, grp = t >> 3;
    const int d = 32 * (p % kLines) + 8 * (m & 3) + dd;
    const int q = row / H, h = row - q * H;
    const int rg = q / kRows, r = q % kRows;
    const size_t item = (size_t)rg * H + h;
    const float2* mlr = pml + (item * kRows + r) * S;
    const float* orow = po + (item * S * kRows + r) * D + d;  // split s: + s * kRows * D
    float M = kInitMax, L = 0.f, A = 0.f;
    for (int base = grp; base < S; base += 8 * kB) {
        float pm[kB], pl[kB], pv[kB];
#pragma unroll
        for (int k = 0; k < kB; ++k) {
            const int s = base + 8 * k;
            const int sc = s < S ? s : base;
            const float2 v = mlr[sc];
            pm[k] = s < S ? v.x : kInitMax;
            pl[k] = v.y;
            pv[k] = orow[(size_t)sc * kRows * D];
        }
        float mb = M;
#pragma unroll
        for (int k = 0; k < kB; ++k) mb = fmaxf(mb, pm[k]);
        // v_exp_f32 without denormal handling: arguments are <= 0 and a weight
        // below 2^-126 of the largest is negligible.
        const float sc = __builtin_amdgcn_exp2f(M - mb);
        L *= sc;
        A *= sc;
#pragma unroll
        for (int k = 0; k < kB; ++k) {
            const float wt = __builtin_amdgcn_exp2f(pm[k] - mb);
            L += pl[k] * wt;
            A += pv[k] * wt;
        }
        M = mb;
    }
    auto merge = [&](float Mp, float Lp, float Ap) {
        const float mn = fmaxf(M, Mp);
        const float a = __builtin_amdgcn_exp2f(M - mn), c = __builtin_amdgcn_exp2f(Mp - mn);
        L = L * a + Lp * c;
        A = A * a + Ap * c;
        M = mn;
    };
    merge(lane_xor<8>(M), lane_xor<8>(L), lane_xor<8>(A));
    merge(lane_xor<16>(M), lane_xor<16>(L), lane_xor<16>(A));
    merge(lane_xor<32>(M), lane_xor<32>(L), lane_xor<32>(A));
    if (t < 8) output[(size_t)row * D + d] = f2h(L > 0.f ? A / L : A);
}

}  // namespace dec

// Paged steps: work segments (workgroups) per CU.
#ifndef TQ_PAGED_SEGMENTS_PER_CU
#define TQ_PAGED_SEGMENTS_PER_CU 1
#endif
constexpr int kPagedSegmentsPerCU = TQ_PAGED_SEGMENTS_PER_CU;

// Slot-mapped decode: the least tokens of a split, and its workgroups per CU.
#ifndef TQ_SPLIT_MIN_TOKENS
#define TQ_SPLIT_MIN_TOKENS 256
#endif
#ifndef TQ_SPLIT_BLOCKS_PER_CU
#define TQ_SPLIT_BLOCKS_PER_CU 2
#endif
constexpr int kSplitMinTokens = TQ_SPLIT_MIN_TOKENS, kSplitBlocksPerCU = TQ_SPLIT_BLOCKS_PER_CU;

bool mfma_attention_ok(const PageGeom& g, const void* pool) {
    const auto al = [](uint64_t v, uint64_t a) { return (v & (a - 1)) == 0; };
    return g.D == 128 && g.code_stride == 64 && al(g.page_size, 16) && al(g.kc_off, 16) &&
           al(g.vc_off, 4) && al(reinterpret_cast<uintptr_t>(pool), 16);
}
// head_dim 64 on the matrix cores: 8-byte K and 2-byte V loads.
bool mfma_attention64_ok(const PageGeom& g, const void* pool) {
    const auto al = [](uint64_t v, uint64_t a) { return (v & (a - 1)) == 0; };
    return g.D == 64 && g.code_stride == 32 && al(g.page_size, 8) && al(g.kc_off, 8) &&
           al(g.vc_off, 2) && al(reinterpret_cast<uintptr_t>(pool), 8);
}

}  // namespace

#define TQ_DISPATCH_D(D_, ...)                                                 \
    switch (D_) {                                                                \
        case 2: { constexpr int kD = 2; __VA_ARGS__; } break;                    \
        case 4: { constexpr int kD = 4; __VA_ARGS__; } break;                    \
        case 8: { constexpr int kD = 8; __VA_ARGS__; } break;                    \
        case 16: { constexpr int kD = 16; __VA_ARGS__; } break;                  \
        case 32: { constexpr int kD = 32; __VA_ARGS__; } break;                  \
        case 64: { constexpr int kD = 64; __VA_ARGS__; } break;                  \
        case 128: { constexpr int kD = 128; __VA_ARGS__; } break;                \
        default: throw Error("head_dim must be a power of two in [2, 128]");     \
    }

namespace {
// The MFMA split-K decode of QJL-1b pages: split + combine launches.
void launch_qjl_mfma(const uint16_t* query, const uint8_t* pool, const int32_t* slots,
                     uint16_t* output, const PageGeom& g, int num_queries, int num_kv_tokens,
                     float inv, hipStream_t stream) {
    const char* split_name = "qjl_fused_attn_split";
    const char* combine_name = "qjl_fused_attn_combine";
    using namespace mfma;
    const int rows = num_queries * g.H;
    const int row_groups = (num_queries + kRows - 1) / kRows;
    const int heads = g.H * row_groups;
    // One 256-token split per workgroup, or longer splits once there are
    // more than ~2 workgroups per CU.
    const int max_splits = std::max(1, (num_kv_tokens + kSplitMinTokens - 1) / kSplitMinTokens);
    const int want = std::max(1, (kSplitBlocksPerCU * num_cus() + heads - 1) / heads);
    int splits = std::min(std::min(max_splits, want), 1024);
    const int tps = num_kv_tokens > 0 ? (num_kv_tokens + splits - 1) / splits : 0;
    if (tps > 0) splits = (num_kv_tokens + tps - 1) / tps;
    const size_t blocks = (size_t)splits * heads;
    float* ws = static_cast<float*>(
        workspace(stream, blocks * kRows * kPartStride * sizeof(float)));
    constexpr int kMaxGridYZ = 65535;
    const dim3 combine_grid = num_queries <= kMaxGridYZ && g.H <= kMaxGridYZ
                                  ? dim3(4, g.H, num_queries)
                                  : dim3(4 * rows);
    if (num_kv_tokens == 0) {  // no partials: the combine writes the zero output
        hipLaunchKernelGGL(attn_mfma_combine_kernel, combine_grid, dim3(256), 0, stream, ws,
                           output, g.H, 0);
        check_launch(combine_name);
        return;
    }
    const dim3 grid = row_groups <= kMaxGridYZ && g.H <= kMaxGridYZ
                          ? dim3(splits, g.H, row_groups)
                          : dim3((unsigned)blocks);
    hipLaunchKernelGGL(qjl::attn_qjl_split_kernel, grid, dim3(64 * qjl::kWaves), 0, stream, query,
                       pool, slots, ws, inv, num_queries, num_kv_tokens, tps, splits, g);
    check_launch(split_name);
    if (splits <= kItemCombineMaxSplits)
        hipLaunchKernelGGL(attn_mfma_combine_items_kernel, dim3(heads), dim3(256), 0, stream,
                           ws, output, g.H, splits, num_queries);
    else
        hipLaunchKernelGGL(attn_mfma_combine_kernel, combine_grid, dim3(256), 0, stream, ws,
                           output, g.H, splits);
    check_launch(combine_name);
}

// The generic split-K decode (attn_partial_kernel + attn_combine_kernel, any
// head_dim and page geometry): one wave per (split, row), enough waves to
// cover the chip several times, at least 32 tokens per split.
struct GenericSplit {
    int splits, tps;
    size_t ws_bytes;
};
GenericSplit generic_split(int rows, int max_tokens, int D) {
    int splits = (2048 + rows - 1) / rows;
    splits = std::min(splits, std::max(1, (max_tokens + 31) / 32));
    splits = std::max(splits, 1);
    const int tps = max_tokens > 0 ? (max_tokens + splits - 1) / splits : 0;
    if (tps > 0) splits = (max_tokens + tps - 1) / tps;
    return {splits, tps, (size_t)splits * rows * (D + 2) * sizeof(float)};
}
// The slot-mapped decode (turbo_prod, turbo_mse; D = 64, 128): split + combine,
// with one row group per workgroup (dec::) or units of up to four that share
// the decoded chunks (unit::).
struct DecodeSplit {
    int rows, row_groups, heads, items, splits, tps;
    bool units;
    long long combine_blocks;
    size_t blocks, ws_bytes, want_bytes;  // want_bytes: room for any call of as many rows and no more tokens
};
// Cost of a split kernel's workgroup: a setup and merge, and a pass of 256
// tokens, in 0.1 us (measured at D = 128, turbo_prod, 2 heads, 250 to 32,768
// tokens, kernel trace: one group 5.9-7.1 us at one pass, 9.8 at two, 14.8 at
// four, 22.5 at eight; a unit of two groups 8.2-9.2 at one, of four 11.6 at
// one, 14.4-15.3 at two, 30.7 at seven).  The same constants serve D = 64,
// turbo_mse and other head counts.  Of 594 shapes of 9 to 256 rows at each D (both
// schemes, 1-8 heads, 64-32,768 tokens, up to 6.3 M rows x heads x tokens) the
// kernel they choose is the faster one or within 5% of it but for 8 at D = 128
// and 7 at D = 64; the worst, 192 rows x 8 heads x 1,143 tokens, takes 18.8 us
// against 12.4 (D = 64: 13.2 against 11.1), since a merge of 1,536 rows costs
// more than kMergeCost.
struct SplitCost {
    int setup, pass;
};
constexpr SplitCost kGroupCost{51, 20}, kPairCost{60, 22}, kUnitCost{78, 33};
// The merge launch, which a single split does without (its kernel writes the
// output: 64-250 tokens 11.8 -> 6.2 us per call, 500 tokens 11.8 -> 7.2-7.6).
constexpr int kMergeCost = 30;
// The split count and its cost: one workgroup runs on a CU at a time, so of
// the counts that fill one to four rounds of the CUs, and one split, the
// cheapest is taken (the fewest splits among equals: the merge reads every
// split's partials).
struct SplitChoice {
    int splits;
    long long cost;
};
SplitChoice choose_splits(int items, int passes, SplitCost c, int cus) {
    const long long whole = ((long long)items + cus - 1) / cus * (c.setup + (long long)c.pass * passes);
    SplitChoice best{1, whole};
    for (int r = 1; r <= 4; ++r) {
        int s = std::min({std::max(1, (int)((long long)r * cus / items)), passes, 1024});
        const int per = (passes + s - 1) / s;
        s = (passes + per - 1) / per;
        const long long rounds = ((long long)items * s + cus - 1) / cus;
        const long long cost =
            rounds * (c.setup + (long long)c.pass * per) + (s > 1 ? kMergeCost : 0);
        if (cost < best.cost || (cost == best.cost && s < best.splits)) best = {s, cost};
    }
    return best;
}
// At head_dim 64 every call leaves room for the most that a slot-mapped call
// takes, 8.7 MB (four rounds of the CUs, up to four row groups each): the kernels
// these replaced fitted nearly every call into the 1 MB that the first one left.
size_t workspace64() { return (size_t)16 * num_cus() * dec::part_bytes(64); }
// What a caller's fixed scratch is held to, whatever the launch takes: at D = 128
// the partials of one 256-token split per workgroup, or of longer splits once
// there are more than ~2 workgroups per CU and row group; at D = 64 the generic
// decode's.
size_t fixed_scratch_bytes(const PageGeom& g, int num_queries, int num_kv_tokens) {
    if (g.D == 64) return generic_split(num_queries * g.H, num_kv_tokens, g.D).ws_bytes;
    const int heads = g.H * ((num_queries + mfma::kRows - 1) / mfma::kRows);
    const int passes = std::max(1, (num_kv_tokens + kSplitMinTokens - 1) / kSplitMinTokens);
    const int want = std::max(1, (kSplitBlocksPerCU * num_cus() + heads - 1) / heads);
    int splits = std::min(std::min(passes, want), 1024);
    const int tps = num_kv_tokens > 0 ? (num_kv_tokens + splits - 1) / splits : 0;
    if (tps > 0) splits = (num_kv_tokens + tps - 1) / tps;
    return (size_t)splits * heads * dec::part_bytes(g.D);
}
DecodeSplit decode_split(const PageGeom& g, int num_queries, int num_kv_tokens) {
    using namespace mfma;
    DecodeSplit d{};
    const int cus = num_cus();
    d.rows = num_queries * g.H;
    d.row_groups = (num_queries + kRows - 1) / kRows;
    d.heads = g.H * d.row_groups;
    // The combine: 32 blocks per 8 (row, 128-byte line) pairs.
    d.combine_blocks = ((long long)d.rows * (g.D / 32) + 7) / 8 * 32;
    const size_t per_split = (size_t)d.heads * dec::part_bytes(g.D);
    const int passes = std::max(1, (num_kv_tokens + kSplitMinTokens - 1) / kSplitMinTokens);
    const int units = g.H * ((d.row_groups + unit::kNP - 1) / unit::kNP);
    // (the splits need not grow with the tokens: 76,800 take 100 where 32,768 take 128)
    d.want_bytes = std::min({passes, 1024, (4 * cus + units - 1) / units}) * per_split;
    if (g.D == 64) d.want_bytes = std::max(d.want_bytes, workspace64());
    const SplitChoice one = choose_splits(d.heads, passes, kGroupCost, cus);
    const SplitChoice un = choose_splits(units, passes, d.row_groups == 2 ? kPairCost : kUnitCost, cus);
    d.units = d.row_groups > 1 && un.cost < one.cost;
    d.items = d.units ? units : d.heads;
    d.splits = d.units ? un.splits : one.splits;
    d.tps = num_kv_tokens > 0 ? (num_kv_tokens + d.splits - 1) / d.splits : 0;
    if (d.tps > 0) d.splits = (num_kv_tokens + d.tps - 1) / d.tps;
    d.blocks = (size_t)d.splits * d.items;
    d.ws_bytes = d.splits * per_split;
    return d;
}
template <int SCH, int D>
void launch_decode_attention(const uint16_t* query, const uint8_t* pool, const int32_t* slots,
                             uint16_t* output, const PageGeom& g, const DecodeSplit& d,
                             int num_queries, int num_kv_tokens, float inv, hipStream_t stream,
                             const char* split_name, const char* combine_name,
                             const Scratch& scratch) {
    using namespace mfma;
    if (d.combine_blocks > INT32_MAX)
        throw Error(std::string(combine_name) + ": too many query rows");
    const int S = num_kv_tokens > 0 ? d.splits : 0;
    char* ws = static_cast<char*>(
        scratch.get(stream, S == 1 ? 0 : d.ws_bytes, split_name, d.want_bytes));
    float* po = reinterpret_cast<float*>(ws);
    float2* pml = reinterpret_cast<float2*>(
        reinterpret_cast<uintptr_t>(ws) + (size_t)d.splits * d.heads * kRows * D * sizeof(float));
    if (num_kv_tokens > 0) {
        constexpr int kMaxGridYZ = 65535;
        const int groups = d.items / g.H;  // row groups, or units of them
        const dim3 grid = groups <= kMaxGridYZ && g.H <= kMaxGridYZ ? dim3(d.splits, g.H, groups)
                                                                    : dim3((unsigned)d.blocks);
        if (d.units)
            hipLaunchKernelGGL((unit::attn_unit_split_kernel<SCH, D, false>), grid,
                               dim3(64 * unit::kWaves), 0, stream, query, pool, slots, po, pml,
                               output, inv, num_queries, num_kv_tokens, d.tps, d.splits, g, PagedRows{});
        else
            hipLaunchKernelGGL((dec::attn_decode_split_kernel<SCH, D>), grid,
                               dim3(64 * dec::kWaves), 0, stream, query, pool, slots, po, pml, output,
                               inv, num_queries, num_kv_tokens, d.tps, d.splits, g);
        check_launch(split_name);
    }
    if (S == 1) return;  // (the split kernel wrote the output)
    // (no partials for an empty context: the combine writes zeros)
    const dim3 cgrid((unsigned)d.combine_blocks);
    if (S <= 16)
        hipLaunchKernelGGL((dec::attn_decode_combine_kernel<D, 2>), cgrid, dim3(64), 0, stream, po,
                           pml, output, g.H, d.rows, S);
    else if (S <= 32)
        hipLaunchKernelGGL((dec::attn_decode_combine_kernel<D, 4>), cgrid, dim3(64), 0, stream, po,
                           pml, output, g.H, d.rows, S);
    else
        hipLaunchKernelGGL((dec::attn_decode_combine_kernel<D, 16>), cgrid, dim3(64), 0, stream, po,
                           pml, output, g.H, d.rows, S);
    check_launch(combine_name);
}

// (generic_split)
template <class Tok>
void launch_generic_attention(Scheme s, const uint16_t* query, const uint8_t* pool, Tok tok,
                              uint16_t* output, const PageGeom& g, int rows,
                              const GenericSplit& sp, float* ws, hipStream_t stream,
                              const char* name) {
    if ((long long)sp.splits * rows > INT32_MAX)
        throw Error(std::string(name) + ": too many query rows");
    const float inv = inv_sqrt_d(g.D);
    const dim3 grid((unsigned)(sp.splits * rows));
    if (s == Scheme::Prod) {
        TQ_DISPATCH_D(g.D, hipLaunchKernelGGL((attn_partial_kernel<kD, true, Tok>), grid, dim3(64),
                                              0, stream, query, pool, tok, ws, g, rows, sp.tps,
                                              sp.splits, inv));
    } else {
        TQ_DISPATCH_D(g.D, hipLaunchKernelGGL((attn_partial_kernel<kD, false, Tok>), grid, dim3(64),
                                              0, stream, query, pool, tok, ws, g, rows, sp.tps,
                                              sp.splits, inv));
    }
    check_launch((std::string(name) + "_partial").c_str());
    TQ_DISPATCH_D(g.D, hipLaunchKernelGGL(attn_combine_kernel<kD>, dim3(rows), dim3(64), 0,
                                          stream, ws, output, g, rows, sp.splits, inv));
    check_launch((std::string(name) + "_combine").c_str());
}

// A paged step on the matrix cores (head_dim 64, 128): the plan, one split
// workgroup per work segment, and a merge per row group and kv head.
template <int SCH, int D>
void launch_paged_units(const uint16_t* query, const uint8_t* pool, const int32_t* block_tables,
                        int max_blocks, const int32_t* row_seq, const int32_t* row_kv_len,
                        uint16_t* output, const PageGeom& g, int num_rows, int max_kv_len,
                        uint64_t extent, hipStream_t stream) {
    using namespace mfma;
    constexpr bool prod = SCH == kSchProd;
    const int row_groups = (num_rows + kRows - 1) / kRows;
    const int heads = g.H * row_groups;
    // The plan gives every kv head the same work (each unit's passes over
    // its kv length), split into Gh equal segments per head, one workgroup
    // each: G = H * Gh workgroups, Gh a multiple of 8 (the kernel's XCD
    // mapping).
    const int Gh = 8 * ((kPagedSegmentsPerCU * num_cus() + 8 * g.H - 1) / (8 * g.H));
    const int G = Gh * g.H;
    // Workspace: the partials (slot (unit + segment) * H + head: fewer than
    // (row_groups + Gh) * H = heads + G slots of kNP positions), then the
    // plan: the units and a sentinel, each row group's unit, the unit count
    // and total work.
    const size_t part_bytes =
        ((size_t)heads + G) * unit::kNP * kRows * unit::part_stride(D) * sizeof(float);
    const size_t unit_bytes = (2 * (size_t)row_groups + 1) * sizeof(PagedUnit);
    const size_t spare_at = (part_bytes + unit_bytes + 4 * sizeof(int32_t) + 255) & ~(size_t)255;
    // head_dim 64: room for the steps of up to 240 (row group, head) pairs, which
    // the kernels these replaced fitted into the least workspace, 1 MB.
    const size_t more = (size_t)std::max(0, 240 - heads) *
                        (unit::kNP * kRows * unit::part_stride(D) * sizeof(float) + 2 * sizeof(PagedUnit));
    char* wsb = static_cast<char*>(workspace(
        stream, spare_at + extent, D == 64 ? std::max(spare_at + extent + more, workspace64()) : 0));
    float* ws = reinterpret_cast<float*>(wsb);
    PagedUnit* units = reinterpret_cast<PagedUnit*>(wsb + part_bytes);
    PagedUnit* group_unit = units + row_groups + 1;
    int32_t* plan = reinterpret_cast<int32_t*>(wsb + part_bytes + unit_bytes);
    // Up to kPlanGroups row groups: each split workgroup makes the plan for
    // itself, its row lengths read in place of the plan's records, and the
    // plan launch (5.5 us of a step) is gone.
    const bool self = row_groups <= unit::kPlanGroups;
    const PagedRows pr{block_tables, row_seq,    row_kv_len, max_blocks, self ? nullptr : units,
                       group_unit,   plan,       reinterpret_cast<const uint8_t*>(wsb + spare_at),
                       0xFFFFFFFFu / (uint32_t)Gh};
    if (!self) {
        hipLaunchKernelGGL(paged_plan_kernel<unit::kNP>, dim3(1), dim3(1024), 0, stream, row_seq,
                           row_kv_len, num_rows, row_groups, unit::kPass, max_kv_len, Gh, units,
                           group_unit, plan);
        check_launch(prod ? "turbo_prod_paged_attn_plan" : "turbo_mse_paged_attn_plan");
    }
    if (max_kv_len > 0 || self) {
        hipLaunchKernelGGL((unit::attn_unit_split_kernel<SCH, D, true>), dim3(G),
                           dim3(64 * unit::kWaves), 0, stream, query, pool, nullptr, ws, nullptr,
                           nullptr, inv_sqrt_d(D), num_rows, max_kv_len, 0, 0, g, pr);
        check_launch(prod ? "turbo_prod_paged_attn_split" : "turbo_mse_paged_attn_split");
    }
    // One wave per row, or per 128-byte line of it while that is few waves.
    const long long lines = (long long)heads * kRows * (D / 32);
    if (lines <= 4096)
        hipLaunchKernelGGL((attn_paged_combine_kernel<D, 8>), dim3((unsigned)lines), dim3(64), 0,
                           stream, ws, output, g.H, num_rows, pr);
    else
        hipLaunchKernelGGL((attn_paged_combine_kernel<D, D / 4>), dim3((unsigned)heads * kRows), dim3(64), 0,
                           stream, ws, output, g.H, num_rows, pr);
    check_launch(prod ? "turbo_prod_paged_attn_combine" : "turbo_mse_paged_attn_combine");
}
}  // namespace

void launch_attention(Scheme s, const uint16_t* query, const uint8_t* pool, const int32_t* slots,
                      uint16_t* output, const PageGeom& g, int num_queries, int num_kv_tokens,
                      hipStream_t stream, const Scratch& scratch) {
    const int rows = num_queries * g.H;
    if (rows <= 0) return;
    const float inv = inv_sqrt_d(g.D);
    const bool prod = s == Scheme::Prod;
    const char* split_name = prod ? "turbo_prod_fused_attn_split" : "turbo_mse_fused_attn_split";
    const char* combine_name =
        prod ? "turbo_prod_fused_attn_combine" : "turbo_mse_fused_attn_combine";
    const bool d64 = mfma_attention64_ok(g, pool);
    if (d64 || mfma_attention_ok(g, pool)) {
        const DecodeSplit d = decode_split(g, num_queries, num_kv_tokens);
        // head_dim 64: where there are too many rows for the combine's grid, the
        // generic decode below takes the call if it can.
        const bool fits = !d64 || (d.combine_blocks <= INT32_MAX && d.blocks <= INT32_MAX);
        if (scratch.ptr)
            scratch.hold(fixed_scratch_bytes(g, num_queries, num_kv_tokens), split_name);
        const auto go = [&](auto sch) {
            constexpr int kSch = decltype(sch)::value;
            if (d64)
                launch_decode_attention<kSch, 64>(query, pool, slots, output, g, d, num_queries,
                                                  num_kv_tokens, inv, stream, split_name,
                                                  combine_name, scratch);
            else
                launch_decode_attention<kSch, 128>(query, pool, slots, output, g, d, num_queries,
                                                   num_kv_tokens, inv, stream, split_name,
                                                   combine_name, scratch);
        };
        if (fits) {
            if (prod)
                go(std::integral_constant<int, mfma::kSchProd>{});
            else
                go(std::integral_constant<int, mfma::kSchMse>{});
            return;
        }
    }
    const GenericSplit sp = generic_split(rows, num_kv_tokens, g.D);
    const char* partial_name = prod ? "turbo_prod_fused_attn_partial" : "turbo_mse_fused_attn_partial";
    scratch.hold(sp.ws_bytes, partial_name);
    float* ws = static_cast<float*>(scratch.get(stream, sp.ws_bytes, partial_name));
    launch_generic_attention(s, query, pool, SlotTokens{slots, num_kv_tokens}, output, g, rows, sp,
                             ws, stream, prod ? "turbo_prod_fused_attn" : "turbo_mse_fused_attn");
}

void launch_paged_attention(Scheme s, const uint16_t* query, const uint8_t* pool,
                            const int32_t* block_tables, int max_blocks, const int32_t* row_seq,
                            const int32_t* row_kv_len, uint16_t* output, const PageGeom& g,
                            int num_rows, int max_kv_len, hipStream_t stream) {
    const int rows = num_rows * g.H;
    if (rows <= 0) return;
    const bool prod = s == Scheme::Prod;
    // Bytes from a page's start that a cell's loads reach (the matrix-core
    // kernel addresses them as 32-bit offsets, and masked tokens read a spare
    // region of this size).
    const uint64_t cells = (uint64_t)g.block_size * (uint64_t)g.H;
    const uint64_t extent =
        std::max({g.page_size, std::max({g.ks_off, g.vs_off, g.kres_off}) + cells * g.scale_stride,
                  std::max(g.kc_off, g.vc_off) + cells * g.code_stride});
    // The plan counts each kv head's work in int32: at most
    // 4 * ceil(max_kv_len / kPass) + kPieceCost per row group (every head has
    // the same).
    const int row_groups = (num_rows + mfma::kRows - 1) / mfma::kRows;
    const bool countable =
        (long long)row_groups *
            (4LL * ((std::max(max_kv_len, 0) + unit::kPass - 1) / unit::kPass) + unit::kPieceCost) <=
        INT32_MAX;
    const bool d64 = mfma_attention64_ok(g, pool) && countable;
    if (!(d64 || mfma_attention_ok(g, pool)) || extent > 0xFFFFFFFFu) {
        // Other head_dims and unaligned pages (and head_dim 64 past the plan's
        // count): the generic split-K decode, its rows reading their tokens
        // through the block table.
        const GenericSplit sp = generic_split(rows, std::max(max_kv_len, 0), g.D);
        float* ws = static_cast<float*>(workspace(stream, sp.ws_bytes));
        launch_generic_attention(
            s, query, pool,
            PagedTokens{block_tables, row_seq, row_kv_len, max_blocks, std::max(max_kv_len, 0)},
            output, g, rows, sp, ws, stream,
            prod ? "turbo_prod_paged_attn" : "turbo_mse_paged_attn");
        return;
    }
    if (!countable) throw Error("paged attention: too many rows for this max_kv_len");
    using namespace mfma;
    const auto go = [&](auto sch, auto dim) {
        launch_paged_units<decltype(sch)::value, decltype(dim)::value>(
            query, pool, block_tables, max_blocks, row_seq, row_kv_len, output, g, num_rows,
            std::max(max_kv_len, 0), extent, stream);
    };
    const auto by_dim = [&](auto sch) {
        if (d64)
            go(sch, std::integral_constant<int, 64>{});
        else
            go(sch, std::integral_constant<int, 128>{});
    };
    if (prod)
        by_dim(std::integral_constant<int, kSchProd>{});
    else
        by_dim(std::integral_constant<int, kSchMse>{});
}

bool launch_qjl_mfma_attention(const uint16_t* query, const uint8_t* pool, const int32_t* slots,
                               uint16_t* output, const QjlGeom& q, int num_queries,
                               int num_kv_tokens, hipStream_t stream) {
    const auto al = [](uint64_t v, uint64_t a) { return (v & (a - 1)) == 0; };
    if (!(q.D == 128 && q.k1_bytes == 16 && q.v4_bytes == 64 && al(q.page_size, 4) &&
          al(q.k1_off, 4) && al(q.v4_off, 4) && al(q.ks_off, 2) && al(q.vs_off, 2) &&
          al(reinterpret_cast<uintptr_t>(pool), 16)))
        return false;
    PageGeom g{};
    g.page_size = q.page_size;
    g.kc_off = q.k1_off;
    g.vc_off = q.v4_off;
    g.ks_off = q.ks_off;
    g.vs_off = q.vs_off;
    g.code_stride = q.v4_bytes;  // V rows; the K sign rows are D/8 = 16 bytes
    g.scale_stride = 2;
    g.H = q.H;
    g.D = q.D;
    g.block_size = q.block_size;
    g.bs_shift = (q.block_size & (q.block_size - 1)) == 0 ? __builtin_ctz(q.block_size) : -1;
    g.h_shift = (q.H & (q.H - 1)) == 0 ? __builtin_ctz(q.H) : -1;
    launch_qjl_mfma(query, pool, slots, output, g, num_queries, num_kv_tokens, inv_sqrt_d(q.D),
                    stream);
    return true;
}

void launch_logits(const uint16_t* query, const uint8_t* pool, const int32_t* slots,
                   float* logits, const PageGeom& g, int num_queries, int num_kv_tokens,
                   hipStream_t stream) {
    const int rows = num_queries * g.H;
    if (rows <= 0 || num_kv_tokens <= 0) return;
    const int tiles = (num_kv_tokens + 255) / 256;
    const float inv = inv_sqrt_d(g.D);
    const int row_groups = (num_queries + 7) / 8;
    if ((g.D == 128 || g.D == 64) && g.code_stride == g.D / 2 && (g.kc_off & 3) == 0 && (g.page_size & 3) == 0 &&
        (g.ks_off & 1) == 0 && (g.kres_off & 1) == 0 &&
        (reinterpret_cast<uintptr_t>(pool) & 3) == 0 && g.H <= 65535 && row_groups <= 65535 &&
        g.page_size <= 0xFFFFFFFFull) {
        const bool vec = (num_kv_tokens & 3) == 0 && (reinterpret_cast<uintptr_t>(logits) & 15) == 0;
        const dim3 grid((num_kv_tokens + lgt::kTokens - 1) / lgt::kTokens, g.H, row_groups);
        const dim3 block(64 * lgt::kWaves);
        const auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, block, 0, stream, query, pool, slots, logits, g,
                               num_queries, num_kv_tokens, inv);
        };
        if (g.D == 128)
            vec ? go(lgt::prod_logits_mfma_kernel<true, 128>) : go(lgt::prod_logits_mfma_kernel<false, 128>);
        else
            vec ? go(lgt::prod_logits_mfma_kernel<true, 64>) : go(lgt::prod_logits_mfma_kernel<false, 64>);
        check_launch("turbo_prod_fused_attention_logits_kernel");
        return;
    }
    TQ_DISPATCH_D(g.D, hipLaunchKernelGGL(prod_logits_kernel<kD>, dim3(rows * tiles), dim3(256),
                                          0, stream, query, pool, slots, logits, g,
                                          num_kv_tokens, tiles, inv));
    check_launch("turbo_prod_fused_attention_logits_kernel");
}

}  // namespace tq
