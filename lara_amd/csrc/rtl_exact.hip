// KV260 RTL-exact numerics mode: the board's bit-level arithmetic on gfx950.
//
// The deployed KV260 datapath does not compute IEEE-exact softmax attention; it computes
// (hw/rtl/pkg/attn_pkg.sv:341-626, hw/rtl/core/softmax_engine.sv:570-1334,
//  hw/rtl/attn_top.sv:653-658, hw/rtl/mem/output_buffer.sv:192-286):
//   S      = sequential fp32 sum over d of exact bf16 products (bf16 exponent 0 reads as 0)
//   s'     = fp32 RNE product with the scale; masked keys -inf
//   per 16-key sub-block and row: row max by bit-pattern compare, m_new = max(m_old, row max),
//   corr   = 0 on the first sub-block, else E(m_old - m_new); p = masked ? 0 : E(s' - m_new),
//   where E is a 1024-entry exp table on [-8, 0] with fixed-point index math and linear
//   interpolation; l = first ? sum p : l*corr + sum p (left to right)
//   dO     = sequential sum over the sub-block's keys of exact products of the UPPER 16 BITS of
//            p (truncation) with V; O = O*corr + dO
//   out    = l == 0 ? 0 : O * R(l), R from a 256-entry reciprocal-mantissa table; bf16 RNE
// over 32-row Q tiles and 64-key KV tiles of four sub-blocks, with the causal KV-tile limit of
// hw/rtl/core/attn_core.sv:138-154.  This kernel reproduces that bit for bit so outputs can be
// compared with board results exactly.
//
// Arithmetic: the RTL's fp32 add and multiply round like IEEE round-to-nearest-even for normal
// operands and results, so the common case runs on native v_add_f32 / v_mul_f32 (with
// contraction off); zero operands, exponent-range edges, inf and NaN take the bit-level path
// that restates the RTL's rules (a zero operand returns the other operand unchanged, 8-bit
// exponent wrap, canonical NaN).
//
// Work decomposition.  What has to run in the board's order is short: the 128-term sum of a score, the
// 16-term sum of a sub-block's O delta, and one fp32 multiply-add per sub-block for l and each O
// element.  Scores of different (row, key) pairs and deltas of different (sub-block, row, dim) are
// independent, so a work-group takes one 32-row tile of one query head and walks its keys 256 at a
// time: every wave computes the scores of 64 keys, the threads then take the exponentials of one
// (row, sub-block) each, and every wave accumulates 32 dims of O.
//
// Both sums run on v_mfma_f32_32x32x1_2b_f32: an outer product with K = 1 is one fused multiply-add per
// result element, rounded to nearest even, and since a product of two bf16 words is exact in fp32
// that is the board's add of an exact product.  A chain of them is the sequential sum, at twice the
// rate of v_fma_f32 and without operand traffic.  It holds while no word, product or partial sum
// leaves the normal range, which words in {0} u [2^-56, 2^34) guarantee (kRangeLo, kRangeHi below); a
// tile with any other word (subnormals, huge values, inf, NaN) takes the bit-level operators.
#include "gqa_internal.h"
#include "rtl_luts.inc"  // kRtlExpLut[1024], kRtlRecipLut[256]: the board's ROM images

#include <math.h>

#include <algorithm>

#pragma clang fp contract(off)

namespace lara {
namespace {

constexpr uint32_t kNan = 0x7FC00000u;
constexpr uint32_t kNegInf = 0xFF800000u;
constexpr uint32_t kOne = 0x3F800000u;
constexpr uint32_t kNegEight = 0xC1000000u;
constexpr int32_t kOrderNegInf = (int32_t)(kNegInf ^ 0x7FFFFFFFu);  // order_word(kNegInf)

__device__ __forceinline__ uint32_t ex(uint32_t a) { return (a >> 23) & 0xFFu; }
__device__ __forceinline__ bool zero_b(uint32_t a) { return (a & 0x7FFFFFFFu) == 0u; }
__device__ __forceinline__ bool nan_b(uint32_t a) { return ex(a) == 0xFFu && (a & 0x7FFFFFu) != 0u; }
__device__ __forceinline__ bool inf_b(uint32_t a) { return ex(a) == 0xFFu && (a & 0x7FFFFFu) == 0u; }
__device__ __forceinline__ bool normal_b(uint32_t a) { return ex(a) - 1u < 254u; }
__device__ __forceinline__ float f_(uint32_t a) { return __uint_as_float(a); }
__device__ __forceinline__ uint32_t b_(float a) { return __float_as_uint(a); }

// ---- bit-level paths (operands or results outside the normal range) ----------------------

__device__ __forceinline__ uint32_t add_bits(uint32_t a, uint32_t b) {
    // 56-bit aligned significands with a sticky bit, leading-zero count limited to 24,
    // round to nearest even, 8-bit exponent arithmetic; exponent 0 reads as 1 without the
    // hidden bit, exponent 255 as an ordinary value.
    const uint32_t ea0 = ex(a), eb0 = ex(b);
    const uint32_t ma = (ea0 ? 0x800000u : 0u) | (a & 0x7FFFFFu);
    const uint32_t mb = (eb0 ? 0x800000u : 0u) | (b & 0x7FFFFFu);
    const uint32_t ea = ea0 ? ea0 : 1u, eb = eb0 ? eb0 : 1u;
    const bool a_big = ea > eb || (ea == eb && ma >= mb);
    const uint32_t e_big = a_big ? ea : eb;
    const uint32_t diff = a_big ? ea - eb : eb - ea;
    const uint64_t big = (uint64_t)(a_big ? ma : mb) << 32;
    const uint64_t small = (uint64_t)(a_big ? mb : ma) << 32;
    uint64_t sh;
    if (diff >= 56u) {
        sh = small != 0 ? 1u : 0u;
    } else {
        sh = small >> diff;
        if (diff != 0u && (small & ((1ull << diff) - 1u)) != 0) sh |= 1u;
    }
    const bool sub = ((a ^ b) >> 31) != 0u;
    const uint64_t sum = sub ? big - sh : big + sh;
    if (sum == 0) return 0u;
    uint32_t e = e_big;
    uint64_t n;
    if (sum >> 56) {
        e = (e + 1u) & 0xFFu;
        n = (sum >> 1) | (sum & 1u);
    } else {
        const uint32_t top = (uint32_t)(sum >> 32) & 0xFFFFFFu;
        const uint32_t lz = top ? (uint32_t)(__clz(top) - 8) : 24u;
        n = (sum << lz) & ((1ull << 56) - 1);
        e = (e - lz) & 0xFFu;
    }
    const uint32_t keep = (uint32_t)(n >> 32) & 0xFFFFFFu;
    const bool guard = (n >> 31) & 1u;
    const bool rest = (n & 0x7FFFFFFFull) != 0;
    uint32_t r = keep + ((guard && (rest || (keep & 1u))) ? 1u : 0u);
    uint32_t frac = r & 0x7FFFFFu;
    if (r >> 24) {
        e = (e + 1u) & 0xFFu;
        frac = 0u;
    }
    return ((a_big ? a : b) & 0x80000000u) | (e << 23) | frac;
}

__device__ __forceinline__ uint32_t mul_bits(uint32_t a, uint32_t b) {
    // both significands carry the hidden bit whatever the exponent; 8-bit exponent wrap
    const uint64_t p = (uint64_t)(0x800000u | (a & 0x7FFFFFu)) * (0x800000u | (b & 0x7FFFFFu));
    const uint32_t top = (uint32_t)(p >> 47) & 1u;
    uint32_t e = (ex(a) + ex(b) - 127u + top) & 0xFFu;
    const uint32_t keep = 0x800000u | ((uint32_t)(p >> (23 + top)) & 0x7FFFFFu);
    const bool guard = (p >> (22 + top)) & 1u;
    const bool rest = (p & ((1ull << (22 + top)) - 1u)) != 0;
    uint32_t r = keep + ((guard && (rest || (keep & 1u))) ? 1u : 0u);
    if (r >> 24) {
        e = (e + 1u) & 0xFFu;
        r = 0x800000u;
    }
    return ((a ^ b) & 0x80000000u) | (e << 23) | (r & 0x7FFFFFu);
}

// ---- the board's operators -------------------------------------------------------------

__device__ __forceinline__ uint32_t add(uint32_t a, uint32_t b) {
    if (normal_b(a) && normal_b(b)) {
        const uint32_t r = b_(f_(a) + f_(b));
        if (normal_b(r)) return r;
        if (r == 0u && a == (b ^ 0x80000000u)) return 0u;  // exact cancellation
        return add_bits(a, b);
    }
    if (nan_b(a) || nan_b(b)) return kNan;
    if (zero_b(a)) return b;
    if (zero_b(b)) return a;
    return add_bits(a, b);
}

__device__ __forceinline__ uint32_t sub(uint32_t a, uint32_t b) { return add(a, b ^ 0x80000000u); }

__device__ __forceinline__ uint32_t mul(uint32_t a, uint32_t b) {
    if (normal_b(a) && normal_b(b)) {
        const uint32_t r = b_(f_(a) * f_(b));
        if (normal_b(r)) return r;
        return mul_bits(a, b);
    }
    if (nan_b(a) || nan_b(b)) return kNan;
    if (zero_b(a) || zero_b(b)) return (a ^ b) & 0x80000000u;
    if (inf_b(a) || inf_b(b)) return ((a ^ b) & 0x80000000u) | 0x7F800000u;
    return mul_bits(a, b);
}

// exact product of two bf16 words
__device__ __forceinline__ uint32_t bmul(uint32_t a16, uint32_t b16) {
    const uint32_t ea = (a16 >> 7) & 0xFFu, eb = (b16 >> 7) & 0xFFu;
    const uint32_t s = ((a16 ^ b16) & 0x8000u) << 16;
    if (ea - 1u < 254u && eb - 1u < 254u && ea + eb - 128u < 253u)  // result exponent 1..254
        return b_(f_(a16 << 16) * f_(b16 << 16));
    const bool az = ea == 0u, bz = eb == 0u;
    const bool ainf = ea == 0xFFu && (a16 & 0x7Fu) == 0u, binf = eb == 0xFFu && (b16 & 0x7Fu) == 0u;
    if ((ea == 0xFFu && !ainf) || (eb == 0xFFu && !binf)) return kNan;
    if ((ainf && bz) || (az && binf)) return kNan;
    if (ainf || binf) return s | 0x7F800000u;
    if (az || bz) return s;
    const uint32_t p = (0x80u | (a16 & 0x7Fu)) * (0x80u | (b16 & 0x7Fu));
    const uint32_t top = p >> 15;
    const uint32_t e = (ea + eb - 127u + top) & 0xFFu;
    return s | (e << 23) | ((p << (9 - top)) & 0x7FFFFFu);
}

// The board compares fp32 words by sign and magnitude, -0 below +0 and NaN by its bits: the order of
// these signed integers (order_word undoes itself).
__device__ __forceinline__ int32_t order_word(uint32_t a) { return (int32_t)(a ^ ((uint32_t)((int32_t)a >> 31) & 0x7FFFFFFFu)); }

// E(x): the interpolated exp table (softmax_engine.sv:570-706), read from its LDS copy.  Below -8 it
// is 0, above 0 it is 1.  On [-8, 0] the Q3.23 magnitude is the truncated |x| * 2^23 (exact: a power of
// two), at most 2^26.  With n its distance from 2^26, the RTL's 36-bit product 1023 n is
// (n / 2^16) 2^26 + t, t = (n % 2^16) 2^10 - n, |t| < 2^26: shifts instead of quarter-rate multiplies.
// The table's steps and its 2^-26 fractions are normal, so native operations round as the RTL's.
__device__ __forceinline__ uint32_t exp_table(const uint32_t* lut, uint32_t x) {
    const uint32_t mag = x & 0x7FFFFFFFu;
    if (!(x >> 31) && mag != 0u) return kOne;
    if (mag > (kNegEight & 0x7FFFFFFFu)) return 0u;
    const uint32_t n = (1u << 26) - (uint32_t)(f_(mag) * 8388608.0f);
    if (n >> 26) return lut[1023];
    const int32_t t = (int32_t)((n & 0xFFFFu) << 10) - (int32_t)n;
    const uint32_t idx = (n >> 16) + (uint32_t)(t >> 31);  // floor(1023 n / 2^26)
    uint32_t rem = (uint32_t)t & 0x3FFFFFFu;
    rem &= rem >> 25 ? ~3u : rem >> 24 ? ~1u : ~0u;  // the fraction's mantissa is truncated to 24 bits
    const float lo = f_(lut[idx]), hi = f_(lut[idx + 1]);
    return b_(lo + (hi - lo) * ((float)rem * 0x1p-26f));
}

// R(l): reciprocal from the mantissa table (output_buffer.sv:192-224)
__device__ __forceinline__ uint32_t recip_table(uint32_t l) {
    const uint32_t s = l & 0x80000000u, e = ex(l), f = l & 0x7FFFFFu;
    if (nan_b(l)) return kNan;
    if (zero_b(l)) return s | 0x7F800000u;
    if (inf_b(l)) return s;
    if (f == 0u) return s | (((254u - e) & 0xFFu) << 23);
    return s | (((253u - e) & 0xFFu) << 23) | kRtlRecipLut[f >> 15];
}

__device__ __forceinline__ uint16_t to_bf16(uint32_t a) {
    const uint32_t up = ((a >> 15) & 1u) && ((a & 0x7FFFu) || ((a >> 16) & 1u));
    return (uint16_t)((a >> 16) + up);
}

typedef float f32x32 __attribute__((ext_vector_type(32)));

constexpr int kTileRows = 32;                  // query rows of a work-group (the board's Q tile)
constexpr int kRtlWaves = 4;
constexpr int kRtlThreads = kRtlWaves * 64;
constexpr int kSpanKeys = kRtlWaves * 64;      // keys of one pass of the work-group
constexpr int kSpanSubs = kSpanKeys / 16;
constexpr int kScoreRow = kSpanKeys + 4;       // LDS row of scores, padded against bank conflicts

// Words whose products and partial sums stay normal: zero, or a bf16 exponent in [71, 160].  Products
// of two such words are multiples of 2^-126 (2 * (71 - 127 - 7)), so a partial sum is zero or normal, and
// below 2^75 (128 products below 2^68), so no sum overflows.  The softmax weights (0, or 2^-12 .. 1) lie within.
constexpr uint32_t kRangeLo = 71u << 7, kRangeHi = (160u << 7) | 0x7Fu;

// Normal values or zero: native operations on them with such a result round as the
// board's (the sign of a zero apart).
__device__ __forceinline__ bool tame_f(float x) { return __builtin_amdgcn_classf(x, 0x168); }

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// Whether a word of N4 16-byte chunks lies outside that range.
template <int N4>
__device__ __forceinline__ bool wild_words(const u32x4 (&w)[N4]) {
    u16x2 lo = {0xFFFF, 0xFFFF}, hi = {0, 0};
#pragma unroll
    for (int i = 0; i < 4 * N4; ++i) {
        const u16x2 a = __builtin_bit_cast(u16x2, w[i >> 2][i & 3] & 0x7FFF7FFFu);
        hi = __builtin_elementwise_max(hi, a);
        lo = __builtin_elementwise_min(lo, (u16x2)(a - (u16x2){1, 1}));  // zero wraps to the largest
    }
    return min((uint32_t)lo.x, (uint32_t)lo.y) < kRangeLo - 1u || max((uint32_t)hi.x, (uint32_t)hi.y) > kRangeHi;
}

// Native operations run unconditionally; where a value of a wave leaves the normal range, that wave redoes
// the step with the bit-level operators, in rolled loops over LDS (they are long).
// One work-group per (32-row tile, query head).  Bound by the vector ALU (about 12 M wave operations and
// 0.59 M outer products of 64 cycles for 512 rows, 32 query heads, D = 128, causal): per score the
// exponential and its subtractions are about 35 operations, per (row, dim) of a sub-block the O update 5.
// That transaction takes 76.6 us of kernel; one lane per row walking its keys alone (256 waves on the
// whole GPU, each sum a chain of dependent adds) took 32.0 ms.
template <int D>
__global__ __launch_bounds__(kRtlThreads, 2) void rtl_transaction_kernel(RtlArgs a) {
    __shared__ __attribute__((aligned(16))) uint32_t s_lds[kTileRows][kScoreRow];  // scores, then weights
    __shared__ uint32_t lut[1024];
    __shared__ int32_t sub_max[kSpanSubs][kTileRows];  // row max of each sub-block (order_word)
    __shared__ uint32_t sub_corr[kSpanSubs][kTileRows];
    __shared__ uint32_t sub_sum[kSpanSubs][kTileRows];
    __shared__ int32_t m_carry[2][kTileRows];  // running max before the pass (by the pass's parity; order_word)
    __shared__ uint32_t l_row[kTileRows];
    __shared__ uint32_t spill[kRtlWaves][2][16][64];  // O and the deltas of a sub-block for the bit-level operators

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, half = lane >> 5;
    const int n_t = (a.q_len + kTileRows - 1) / kTileRows;
    const int lin = (int)(blockIdx.y * gridDim.x + blockIdx.x);  // heads fastest
    if (lin >= n_t * a.n_q_heads) return;
    const int hq = lin % a.n_q_heads, by = lin / a.n_q_heads;
    // Row tile: longest first, or, in a grid that is resident at once (two work-groups per CU), the
    // shortest beside the longest (512 rows x 32 heads, causal: 76.6 us against 81.9).
    const int t = a.pair_tiles && by >= (n_t + 1) / 2 ? by - (n_t + 1) / 2 : n_t - 1 - by;
    const int hk = hq / (a.n_q_heads / a.n_kv_heads);
    const uint16_t* kb = a.kc + (size_t)hk * a.l_cap * D;
    const uint16_t* vb = a.vc + (size_t)hk * a.l_cap * D;
    const uint16_t* qb = a.q + ((size_t)hq * a.q_len + kTileRows * t) * D;
    const int rows = min(kTileRows, a.q_len - kTileRows * t);

    // Sub-blocks of the tile's walk.
    const int q_end = a.q_pos_base + kTileRows * t + rows - 1;
    const int n_kv_tiles = (a.kv_len + 63) / 64;
    int last_tile = n_kv_tiles - 1;
    if (a.causal) last_tile = q_end < a.kv_pos_base ? 0 : min((q_end - a.kv_pos_base) / 64, n_kv_tiles - 1);
    const int n_subs = min((last_tile + 1) * 4, (a.kv_len + 15) / 16);

    for (int i = tid; i < 1024; i += kRtlThreads) lut[i] = kRtlExpLut[i];
    if (tid < kTileRows) m_carry[0][tid] = kOrderNegInf;

    const bool has_dims = wave * 32 < D;  // the wave's 32 dims of O
    float o[16];                          // O of row `col`, dims 32 wave + 8 (i/4) + 4 half + i%4
#pragma unroll
    for (int i = 0; i < 16; ++i) o[i] = 0.f;
    bool o_wild = false;  // O has taken words outside the range: only the bit-level operators from then on
    // O holds a word of exponent 255, which only the bit-level operators make (a product's exponent that wraps):
    // native operations would read it as infinite or NaN.
    bool o_past = false;
    uint32_t l = 0u;      // of row `col` (wave 3)
    const float scale = f_(a.scale_bits);
    // Scores are zero or at least 2^-126, so with such a scale only a zero one has a zero product natively; under a
    // smaller one a product may vanish where the board's exponent wraps.
    const bool scale_native = normal_b(a.scale_bits) && scale >= 0x1p-23f;

    for (int sub0 = 0, pass = 0; sub0 < n_subs; sub0 += kSpanSubs, ++pass) {
        const int key0 = sub0 * 16;
        const int subs = min(kSpanSubs, n_subs - sub0);

        // ---- scaled scores of 64 keys per wave (lane: key for the K words, row for the Q words) ----
        const int wkey0 = key0 + 64 * wave;
        if (64 * wave < 16 * subs) {
            const bool in_k = wkey0 + lane < a.kv_len, in_q = col < rows;
            const u32x4* kr = reinterpret_cast<const u32x4*>(kb + (size_t)(in_k ? wkey0 + lane : 0) * D);
            const u32x4* qr = reinterpret_cast<const u32x4*>(qb + (size_t)(in_q ? col : 0) * D);
            constexpr int kPart = 4;  // 16-byte loads of a row in flight
            u32x4 kw[kPart], qw[kPart];
            auto load_kq = [&](int p) {
#pragma unroll
                for (int i = 0; i < kPart; ++i) {
                    kw[i] = in_k ? kr[p * kPart + i] : u32x4{0u, 0u, 0u, 0u};
                    qw[i] = in_q ? qr[p * kPart + i] : u32x4{0u, 0u, 0u, 0u};
                }
            };
            bool wild = false;
            f32x32 acc;  // keys wkey0 + 32 (i/16) + 8 (i/4 % 4) + 4 half + i%4 of row `col`
#pragma unroll
            for (int i = 0; i < 32; ++i) acc[i] = 0.f;
            load_kq(0);
#pragma unroll 1
            for (int p = 0; p < D / (8 * kPart); ++p) {
                u32x4 kc[kPart], qc[kPart];
#pragma unroll
                for (int i = 0; i < kPart; ++i) {
                    kc[i] = kw[i];
                    qc[i] = qw[i];
                }
                if ((p + 1) * 8 * kPart < D) load_kq(p + 1);
                wild |= wild_words(kc) || wild_words(qc);
#pragma unroll
                for (int i = 0; i < 4 * kPart; ++i) {
                    const uint32_t k2 = kc[i >> 2][i & 3], q2 = qc[i >> 2][i & 3];
                    acc = __builtin_amdgcn_mfma_f32_32x32x1f32(f_(k2 << 16), f_(q2 << 16), acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x1f32(f_(k2 & 0xFFFF0000u), f_(q2 & 0xFFFF0000u), acc, 0, 0, 0);
                }
            }
            if (__ballot(wild) == 0) {
                if (pass > 0) __syncthreads();  // the last pass's weights are read
                bool tame = true;
#pragma unroll
                for (int i = 0; i < 32; ++i) tame &= tame_f(acc[i] * scale);
                tame = scale_native && __ballot(!tame) == 0;
                const float by = tame ? scale : 1.f;
#pragma unroll
                for (int i4 = 0; i4 < 8; ++i4)
                    *reinterpret_cast<float4*>(&s_lds[col][64 * wave + 32 * (i4 >> 2) + 8 * (i4 & 3) + 4 * half]) =
                        make_float4(acc[4 * i4] * by, acc[4 * i4 + 1] * by, acc[4 * i4 + 2] * by, acc[4 * i4 + 3] * by);
                if (!tame) {
#pragma unroll 1
                    for (int k = 0; k < 32; ++k) {
                        uint32_t& w = s_lds[col][64 * wave + 2 * k + half];
                        w = mul(w, a.scale_bits);
                    }
                }
            } else {
                if (pass > 0) __syncthreads();
#pragma unroll 1
                for (int r = 0; r < kTileRows; ++r) {
                    uint32_t acc = 0u;
                    if (r < rows && in_k) {
                        const uint32_t* qp = reinterpret_cast<const uint32_t*>(qb + (size_t)r * D);
                        const uint32_t* kp = reinterpret_cast<const uint32_t*>(kr);
#pragma unroll 1
                        for (int d = 0; d < D; ++d)
                            acc = add(acc, bmul(qp[d >> 1] >> (16 * (d & 1)) & 0xFFFFu,
                                                kp[d >> 1] >> (16 * (d & 1)) & 0xFFFFu));
                    }
                    s_lds[r][64 * wave + lane] = mul(acc, a.scale_bits);
                }
            }
        } else if (pass > 0) {
            __syncthreads();
        }
        __syncthreads();

        // ---- softmax of one (row, sub-block) per thread and step ----
        const int r = tid & (kTileRows - 1);
        const int q_pos = a.q_pos_base + kTileRows * t + r;
        const int n_keys = a.causal ? min(a.kv_len, q_pos - a.kv_pos_base + 1) : a.kv_len;  // the row attends 0 .. n_keys-1
#pragma unroll 1
        for (int s = tid >> 5; s < subs; s += kRtlThreads / kTileRows) {
            const int n_live = n_keys - (key0 + 16 * s);
            int32_t mxv = kOrderNegInf;
#pragma unroll
            for (int c4 = 0; c4 < 4; ++c4) {
                const u32x4 sc = *reinterpret_cast<const u32x4*>(&s_lds[r][16 * s + 4 * c4]);
#pragma unroll
                for (int j = 0; j < 4; ++j) mxv = max(mxv, 4 * c4 + j < n_live ? order_word(sc[j]) : kOrderNegInf);
            }
            sub_max[s][r] = mxv;
        }
        __syncthreads();
#pragma unroll 1
        for (int s = tid >> 5; s < subs; s += kRtlThreads / kTileRows) {
            const int n_live = n_keys - (key0 + 16 * s);
            int32_t before = m_carry[pass & 1][r];
#pragma unroll
            for (int i = 0; i < kSpanSubs - 1; ++i) before = max(before, i < s ? sub_max[i][r] : kOrderNegInf);
            const int32_t after = max(before, sub_max[s][r]);
            if (s == subs - 1) m_carry[(pass + 1) & 1][r] = after;
            const uint32_t m_new = (uint32_t)order_word((uint32_t)after);
            sub_corr[s][r] = sub0 + s == 0 ? 0u : exp_table(lut, sub((uint32_t)order_word((uint32_t)before), m_new));
            u32x4 w[4];
            bool tame = tame_f(f_(m_new));
            float sum = 0.f;
#pragma unroll
            for (int c4 = 0; c4 < 4; ++c4) {
                w[c4] = *reinterpret_cast<const u32x4*>(&s_lds[r][16 * s + 4 * c4]);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const bool live = 4 * c4 + j < n_live;
                    const float x = f_(w[c4][j]) - f_(m_new);
                    tame &= !live || (tame_f(f_(w[c4][j])) && tame_f(x));
                    const uint32_t p = live ? exp_table(lut, b_(x)) : 0u;
                    sum += f_(p);                // weights are 0 or normal, and so are their sums
                    w[c4][j] = p & 0xFFFF0000u;  // the PV product takes the upper half of p (truncation)
                }
            }
            if (n_live > 0 && !tame) {
                sum = 0.f;
#pragma unroll 1
                for (int c = 0; c < 16; ++c) {
                    uint32_t& v = s_lds[r][16 * s + c];
                    const uint32_t p = c < n_live ? exp_table(lut, sub(v, m_new)) : 0u;
                    sum += f_(p);
                    v = p & 0xFFFF0000u;
                }
            } else {
#pragma unroll
                for (int c4 = 0; c4 < 4; ++c4) *reinterpret_cast<u32x4*>(&s_lds[r][16 * s + 4 * c4]) = w[c4];
            }
            sub_sum[s][r] = b_(sum);
        }
        __syncthreads();

        // ---- l (wave 3), and O: the deltas of two sub-blocks per chain of 16 outer products ----
        if (wave == kRtlWaves - 1) {
#pragma unroll 1
            for (int s = 0; s < subs; ++s)
                l = sub0 + s == 0 ? sub_sum[s][col] : add(mul(l, sub_corr[s][col]), sub_sum[s][col]);
        }
        if (has_dims) {
            uint32_t vw[16];  // V of the next two sub-blocks: sub-block `half`, dim 32 wave + col
            auto load_v = [&](int s2) {
                const int k0 = key0 + 16 * (s2 + half);
                const uint16_t* vp = vb + (size_t)k0 * D + 32 * wave + col;
                if (s2 + 2 <= subs && key0 + 16 * s2 + 32 <= a.kv_len) {
#pragma unroll
                    for (int c = 0; c < 16; ++c) vw[c] = vp[c * D];
                    return;
                }
#pragma unroll
                for (int c = 0; c < 16; ++c) {
                    vw[c] = 0u;
                    if (s2 + half < subs && k0 + c < a.kv_len) vw[c] = vp[c * D];
                }
            };
            load_v(0);
            for (int s2 = 0; s2 < subs; s2 += 2) {
                float vf[16];
                u32x4 packed[2];
#pragma unroll
                for (int c = 0; c < 16; ++c) {
                    vf[c] = f_(vw[c] << 16);
                    if (c & 1) packed[c >> 3][(c >> 1) & 3] = vw[c - 1] | b_(vf[c]);
                }
                o_wild = o_wild || __ballot(wild_words(packed)) != 0;
                if (s2 + 2 < subs) load_v(s2 + 2);
                const uint32_t* prow = &s_lds[col][16 * s2];  // weights of the pair's 32 keys
                f32x32 acc;  // deltas: sub-block i/16, dim 8 (i/4 % 4) + 4 half + i%4
#pragma unroll
                for (int i = 0; i < 32; ++i) acc[i] = 0.f;
                if (!o_wild) {
#pragma unroll
                    for (int c = 0; c < 16; ++c) acc = __builtin_amdgcn_mfma_f32_32x32x1f32(vf[c], f_(prow[16 * half + c]), acc, 0, 0, 0);
                }
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const int s = s2 + e;
                    if (s >= subs) break;
                    const float corr = f_(sub_corr[s][col]);
                    float r16[16];
                    float least = 1.f;  // zero and subnormal values take the bit-level operators
                    if (sub0 + s == 0) {
#pragma unroll
                        for (int i = 0; i < 16; ++i) {
                            r16[i] = acc[16 * e + i];
                            least = fminf(least, fabsf(r16[i]));
                        }
                    } else {
#pragma unroll
                        for (int i = 0; i < 16; ++i) {
                            const float scaled = o[i] * corr;
                            r16[i] = scaled + acc[16 * e + i];
                            least = fminf(least, fminf(fabsf(scaled), fabsf(r16[i])));
                        }
                    }
                    if (!o_wild && !o_past && __ballot(least < 0x1p-126f) == 0) {
#pragma unroll
                        for (int i = 0; i < 16; ++i) o[i] = r16[i];
                        continue;
                    }
                    const int c0 = key0 + 16 * s;
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        spill[wave][0][i][lane] = b_(o[i]);
                        spill[wave][1][i][lane] = b_(acc[16 * e + i]);
                    }
#pragma unroll 1
                    for (int i = 0; i < 16; ++i) {
                        const int d = 32 * wave + 8 * (i >> 2) + 4 * half + (i & 3);
                        uint32_t delta = spill[wave][1][i][lane];
                        if (o_wild || zero_b(delta)) {  // (a zero delta has the sign of its last product)
                            delta = 0u;
#pragma unroll 1
                            for (int c = 0; c < 16; ++c) {
                                const uint32_t w = c0 + c < a.kv_len ? vb[(size_t)(c0 + c) * D + d] : 0u;
                                delta = add(delta, bmul(prow[16 * e + c] >> 16, w));
                            }
                        }
                        spill[wave][0][i][lane] = add(mul(spill[wave][0][i][lane], b_(corr)), delta);
                    }
                    bool past = false;
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        o[i] = f_(spill[wave][0][i][lane]);
                        past |= ex(b_(o[i])) == 255u;
                    }
                    o_past = __ballot(past) != 0;
                }
            }
        }
    }

    if (wave == kRtlWaves - 1 && half == 0) l_row[col] = l;
    __syncthreads();
    if (col >= rows) return;
    const uint32_t lr = l_row[col];
    if (has_dims) {
        uint16_t* orow = a.out + ((size_t)hq * a.q_len + kTileRows * t + col) * D + 32 * wave + 4 * half;
        const uint32_t rl = recip_table(lr);
#pragma unroll
        for (int i = 0; i < 16; ++i) spill[wave][0][i][lane] = b_(o[i]);
#pragma unroll 1
        for (int i4 = 0; i4 < 4; ++i4) {
            uint32_t w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] = zero_b(lr) ? 0u : to_bf16(mul(spill[wave][0][4 * i4 + j][lane], rl));
            *reinterpret_cast<uint2*>(orow + 8 * i4) = make_uint2(w[0] | (w[1] << 16), w[2] | (w[3] << 16));
        }
    }
    if (a.lse != nullptr && wave == 0 && half == 0) {
        // natural-log LSE of the board's (m, l): m is in scaled-score units
        const int passes = (n_subs + kSpanSubs - 1) / kSpanSubs;
        a.lse[(size_t)hq * a.q_len + kTileRows * t + col] =
            zero_b(lr) ? -INFINITY : f_((uint32_t)order_word((uint32_t)m_carry[passes & 1][col])) + logf(f_(lr));
    }
}

}  // namespace

hipError_t launch_rtl_transaction(int head_dim, const RtlArgs& args, int n_cu, const Launch& l) {
    RtlArgs a = args;
    // The (tile, head) pairs in rows of at most 2^16 work-groups (an axis of the grid holds 2^32 threads, y and z 65535
    // work-groups).
    const int64_t pairs = (int64_t)a.n_q_heads * ((a.q_len + kTileRows - 1) / kTileRows);
    const int64_t per_row = std::min<int64_t>(pairs, 1 << 16), rows = (pairs + per_row - 1) / per_row;
    if (pairs + per_row > INT32_MAX) return hipErrorInvalidValue;
    const dim3 grid((unsigned)per_row, (unsigned)rows), block(kRtlThreads);
    a.pair_tiles = pairs <= 2 * (int64_t)n_cu;
    if (head_dim == 128) return launch_kernel(rtl_transaction_kernel<128>, grid, block, l, a);
    if (head_dim == 64) return launch_kernel(rtl_transaction_kernel<64>, grid, block, l, a);
    return hipErrorInvalidValue;
}

}  // namespace lara
