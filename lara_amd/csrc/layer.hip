// Layer input stage of run_layer (sw/attn_driver.py:552-576): the host RMSNorm, RoPE and
// head reshaping that the reference does in numpy before each attention transaction, here
// as two small HBM-bound kernels around the QKV projection GEMM.
//
// rms_norm_*_kernel: y = x / sqrt(mean(x^2) + eps) * gamma per token row
//   (hw/rtl/ext/rms_norm/rms_norm.sv:7-8, 42-45: sum of squares, inverse square root, two
//   products), sums and products in fp32, one RNE rounding to bf16.  The same launch fills the
//   RoPE cos/sin table in extra work-groups: the norm is memory-bound, so the double-precision
//   sin/cos run on otherwise idle ALUs, off the RoPE kernel's path.
// rope_scatter_kernel: rotation of each (2p, 2p+1) pair of a Q or K head by
//   pos * theta[p] (hw/rtl/core/rope_engine.sv:4-10, 135-155: phase = fp32(pos * theta), then
//   a*cos - b*sin and a*sin + b*cos, each product and sum rounded to fp32), cos/sin of the
//   fp32 phase evaluated in double and rounded to fp32, output rounded to bf16 (RNE).  Q is
//   written head-major [H_q][n_tokens][D] (reshape_to_heads), K and V rows go straight into
//   the sequence's cache rows.
#include "gqa_internal.h"

#include <algorithm>
#include <type_traits>

namespace lara {
namespace {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float bf16_to_f32(uint32_t w) { return __uint_as_float(w << 16); }

constexpr int kNormThreads = 256;

constexpr int kNormCached = 4;  // 16-byte chunks a thread keeps in registers (hidden <= 8192)

__host__ __device__ inline bool norm_vectorised(const NormArgs& a) {
    return (a.hidden & 7) == 0 &&
           ((reinterpret_cast<uintptr_t>(a.x) | reinterpret_cast<uintptr_t>(a.gamma) | reinterpret_cast<uintptr_t>(a.y)) &
            15) == 0;
}

__device__ __forceinline__ float sum_squares(const u32x4& w) {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float lo = bf16_to_f32(w[j] & 0xFFFFu), hi = bf16_to_f32(w[j] >> 16);
        ss += lo * lo;
        ss += hi * hi;
    }
    return ss;
}

__device__ __forceinline__ u32x4 scale_row(const u32x4& w, const u32x4& g, float inv) {
    u32x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float lo = __fmul_rn(__fmul_rn(bf16_to_f32(w[j] & 0xFFFFu), inv), bf16_to_f32(g[j] & 0xFFFFu));
        const float hi = __fmul_rn(__fmul_rn(bf16_to_f32(w[j] >> 16), inv), bf16_to_f32(g[j] >> 16));
        const bf16x2_t pair = {(__bf16)lo, (__bf16)hi};  // v_cvt_pk_bf16_f32, round to nearest even
        o[j] = __builtin_bit_cast(uint32_t, pair);
    }
    return o;
}

// (cos, sin) of the fp32 phase pos * theta, evaluated in double.
__device__ __forceinline__ float2 rope_cos_sin(int pos, float theta) {
#pragma clang fp contract(off)
    double sd, cd;
    sincos((double)((float)pos * theta), &sd, &cd);
    return make_float2((float)cd, (float)sd);
}

// Work-group `wg` (< table_wgs) of a norm launch: one table entry per thread.
__device__ __forceinline__ void fill_rope_table(const RopeTable& t, int wg) {
    const int i = wg * kNormThreads + threadIdx.x;
    if (i >= t.sets * t.n_tokens * t.pairs) return;
    const int p = i % t.pairs, tok = (i / t.pairs) % t.n_tokens, set = i / (t.pairs * t.n_tokens);
    reinterpret_cast<float2*>(t.cs)[i] = rope_cos_sin((set ? t.kv_pos_base : t.q_pos_base) + tok, t.theta[p]);
}

// Row-per-wave form for hidden = CPL * 512 (16-byte aligned rows): each wave owns one token
// row, holds its CPL chunks of x and of gamma in registers (chunk c * 64 + lane, so every load
// instruction covers 1 KiB of the row), sums the squares with a wave reduction (no LDS, no
// barrier) and writes the scaled row.  Rows are independent, so a wave whose loads return
// early computes and stores while other waves' loads are still in flight.
template <int CPL>
__global__ __launch_bounds__(kNormThreads) void rms_norm_wave_kernel(NormArgs a) {
    if ((int)blockIdx.x < a.table_wgs) {
        fill_rope_table(a.table, blockIdx.x);
        return;
    }
    const int lane = threadIdx.x & 63;
    const int row = (blockIdx.x - a.table_wgs) * (kNormThreads / 64) + (threadIdx.x >> 6);
    if (row >= a.n_tokens) return;
    const u32x4* x = reinterpret_cast<const u32x4*>(a.x + (size_t)row * a.hidden);
    const u32x4* g = reinterpret_cast<const u32x4*>(a.gamma);
    u32x4 v[CPL], gv[CPL];
#pragma unroll
    for (int c = 0; c < CPL; ++c) v[c] = __builtin_nontemporal_load(x + c * 64 + lane);
#pragma unroll
    for (int c = 0; c < CPL; ++c) gv[c] = g[c * 64 + lane];
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < CPL; ++c) ss += sum_squares(v[c]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
    const float inv = 1.0f / sqrtf(ss / (float)a.hidden + a.eps);
    u32x4* y = reinterpret_cast<u32x4*>(a.y + (size_t)row * a.hidden);
#pragma unroll
    for (int c = 0; c < CPL; ++c) y[c * 64 + lane] = scale_row(v[c], gv[c], inv);  // the projection reads y next
}

// General form: one work-group per token row.  With hidden % 8 == 0 and 16-byte aligned rows each
// thread moves 16-byte chunks and keeps its first kNormCached chunks in registers between the sum
// of squares and the scaling pass; otherwise one bf16 per thread and step.  With gamma == nullptr
// the launch only fills the table.
__global__ __launch_bounds__(kNormThreads) void rms_norm_kernel(NormArgs a) {
    if ((int)blockIdx.x < a.table_wgs) {
        fill_rope_table(a.table, blockIdx.x);
        return;
    }
    const int row = blockIdx.x - a.table_wgs;
    const uint16_t* x = a.x + (size_t)row * a.hidden;
    uint16_t* y = a.y + (size_t)row * a.hidden;
    const bool vec = norm_vectorised(a);
    constexpr int kStep = kNormThreads * 8;
    float ss = 0.f;
    u32x4 cache[kNormCached], gcache[kNormCached];  // x and gamma chunks, gamma loaded with x
    if (vec) {
#pragma unroll
        for (int c = 0; c < kNormCached; ++c) {
            const int i = c * kStep + threadIdx.x * 8;
            cache[c] = i < a.hidden ? __builtin_nontemporal_load((const u32x4*)(x + i)) : u32x4{0u, 0u, 0u, 0u};
            gcache[c] = i < a.hidden ? *(const u32x4*)(a.gamma + i) : u32x4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int c = 0; c < kNormCached; ++c) ss += sum_squares(cache[c]);
        for (int i = kNormCached * kStep + threadIdx.x * 8; i < a.hidden; i += kStep)
            ss += sum_squares(*(const u32x4*)(x + i));
    } else {
        for (int i = threadIdx.x; i < a.hidden; i += kNormThreads) {
            const float f = bf16_to_f32(x[i]);
            ss += f * f;
        }
    }
    // Wave sum, then the four waves through LDS.
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
    __shared__ float part[kNormThreads / 64];
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
    __syncthreads();
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < kNormThreads / 64; ++w) total += part[w];
    const float inv = 1.0f / sqrtf(total / (float)a.hidden + a.eps);
    if (vec) {
#pragma unroll
        for (int c = 0; c < kNormCached; ++c) {
            const int i = c * kStep + threadIdx.x * 8;
            if (i < a.hidden) *(u32x4*)(y + i) = scale_row(cache[c], gcache[c], inv);
        }
        for (int i = kNormCached * kStep + threadIdx.x * 8; i < a.hidden; i += kStep)
            *(u32x4*)(y + i) = scale_row(*(const u32x4*)(x + i), *(const u32x4*)(a.gamma + i), inv);
    } else {
        for (int i = threadIdx.x; i < a.hidden; i += kNormThreads)
            y[i] = f32_to_bf16_rne(__fmul_rn(__fmul_rn(bf16_to_f32(x[i]), inv), bf16_to_f32(a.gamma[i])));
    }
}

constexpr int kRopeThreads = 256;

// Rotates the pair (x0, x1) of bf16 words; each product and sum is rounded to fp32 on its own.
__device__ __forceinline__ uint32_t rotate_pair(uint32_t x0w, uint32_t x1w, float c, float s) {
#pragma clang fp contract(off)
    const float x0 = bf16_to_f32(x0w), x1 = bf16_to_f32(x1w);
    const float r0 = x0 * c - x1 * s;
    const float r1 = x0 * s + x1 * c;
    return (uint32_t)f32_to_bf16_rne(r0) | ((uint32_t)f32_to_bf16_rne(r1) << 16);
}

// The K (or V) cache row of kv head g for token t; nullptr where its page is unmapped (nothing to write).
__device__ __forceinline__ uint16_t* cache_row(const RopeArgs& a, bool is_k, int g, int t) {
    int64_t r = (int64_t)g * a.l_cap + a.row0 + t;
    if (a.block_table != nullptr) r = paged_row(a.block_table, a.page_shift, a.n_kv_heads, g, a.row0 + t);
    return r < 0 ? nullptr : (is_k ? a.kc : a.vc) + (size_t)r * a.head_dim;
}

// Rotate the four (2p, 2p+1) pairs of one 16-byte chunk of head h by the (cos, sin) values cs
// (two pairs per float4) and store the chunk at its destination.
__device__ __forceinline__ void rope_store_chunk(const RopeArgs& a, int t, int h, int cw, u32x4 w, const float4* cq,
                                                 const float4* ck) {
    const int D = a.head_dim;
    const bool is_q = h < a.n_q_heads, is_k = !is_q && h < a.n_q_heads + a.n_kv_heads;
    if (a.rope && (is_q || is_k)) {
        const float4* csp = is_q ? cq : ck;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float4 pair2 = csp[j >> 1];
            const float c = (j & 1) ? pair2.z : pair2.x, s = (j & 1) ? pair2.w : pair2.y;
            w[j] = rotate_pair(w[j] & 0xFFFFu, w[j] >> 16, c, s);
        }
    }
    uint16_t* dst = is_q ? a.q_out + ((size_t)h * a.n_tokens + t) * D
                         : cache_row(a, is_k, is_k ? h - a.n_q_heads : h - a.n_q_heads - a.n_kv_heads, t);
    if (dst != nullptr) *reinterpret_cast<u32x4*>(dst + 8 * cw) = w;
}

// One work-group per token: the token's H_q + 2 H_kv head rows move in 16-byte chunks of four
// (2p, 2p+1) pairs, one chunk per thread and step (three steps for a 32 + 2 x 8 head, D = 128
// token; 128, 512 and 768 threads measured slower at 2048 tokens).  kRopeThreads is a multiple of
// D / 8, so a thread's pairs are the same in every head: it loads their cos/sin from the table
// once per position set.  No LDS and no barrier: every chunk streams independently.
__global__ __launch_bounds__(kRopeThreads) void rope_scatter_kernel(RopeArgs a) {
    const int t = blockIdx.x;
    const int D = a.head_dim, P = D / 2, CPH = D / 8;  // pairs and 16-byte chunks per head row
    const int n_chunks = (a.n_q_heads + 2 * a.n_kv_heads) * CPH;
    const int cw = threadIdx.x % CPH;
    const u32x4* src = reinterpret_cast<const u32x4*>(a.qkv + (size_t)t * a.ld);
    float4 cq[2] = {}, ck[2] = {};  // (cos, sin) of pairs 4cw .. 4cw+3 at the Q and the K position
    if (a.rope) {
        const float4* tq = reinterpret_cast<const float4*>(a.cs + ((size_t)t * P + 4 * cw) * 2);
        cq[0] = tq[0];
        cq[1] = tq[1];
        const float4* tk = reinterpret_cast<const float4*>(a.cs + (((size_t)a.cs_k_set * a.n_tokens + t) * P + 4 * cw) * 2);
        ck[0] = tk[0];
        ck[1] = tk[1];
    }
    for (int ci = threadIdx.x; ci < n_chunks; ci += kRopeThreads)
        rope_store_chunk(a, t, ci / CPH, cw, __builtin_nontemporal_load(src + ci), cq, ck);
}

// ---- the whole stage for few tokens -------------------------------------------------------------

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kTileOut = 16;  // output rows (of W) of a tile, and the most tokens of a call
constexpr int kFewWaves = 8;

// Tokens whose normalised rows fit the LDS beside the rest (16 columns of the MFMA; more tokens go to the
// library product).
constexpr int few_tokens_most(int hidden) { return hidden > 4096 ? 8 : 16; }

// Sum over the wave, in every lane: lane exchanges within 16 lanes, then across them.
__device__ __forceinline__ float wave_sum(float x) {
    auto add = [](float v, auto ctrl) {
        return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), decltype(ctrl)::value, 0xF, 0xF, true));
    };
    x = add(x, std::integral_constant<int, 0xB1>{});   // quad_perm [1, 0, 3, 2]
    x = add(x, std::integral_constant<int, 0x4E>{});   // quad_perm [2, 3, 0, 1]
    x = add(x, std::integral_constant<int, 0x141>{});  // row_half_mirror
    x = add(x, std::integral_constant<int, 0x140>{});  // row_mirror
    return pair_sum32(pair_sum16(x));
}

// RMSNorm, projection, RoPE and scatter of a few tokens in one launch.  The stage is then the weights'
// stream (48 MiB at hidden 4096 and 6144 outputs), and the launches around a library product cost as
// much as half of it.  One work-group per CU takes output tiles of 16 rows in turn; its waves split
// `hidden` and run v_mfma_f32_16x16x32_bf16 (A: 16 rows of W, straight from memory; B: the normalised
// tokens, from LDS).  Two chunks of R loads each (256 KiB per CU) are in flight from the first
// instructions on, across tiles, behind the loads of x only, which the norm waits for; the norm and
// the rotations are done while the first weights arrive.  The waves' partial products meet in LDS.
// us a launch on one stream / over three, back to back over 1 GiB of weight sets (more than any cache holds), norm,
// library product and RoPE against this: hidden 4096, 32/8 heads of 128 (a streaming read of the weights alone 8.7):
// one token 19.0 / 16.6 against 15.3 / 12.7, 4: 19.7 / 16.4 against 15.8 / 11.6, 16: 21.7 / 16.2 against 19.2 / 14.7;
// hidden 2048, 16/8 heads (4.2): 16.6 / 16.1 against 7.3 / 5.7 (one) .. 10.2 / 8.6 (16); hidden 8192, 64/8 heads
// (25.3): 41.8 / 31.1 against 37.9 / 28.9 (one) .. 43.2 / 32.9 against 41.2 / 32.1 (8).
// (Two resident 16-row work-groups per CU with their own norms, one token over three streams: 14.0, 5.3 and 48.3.)
template <int HIDDEN>
struct FewTokensLds {
    static constexpr int kRow = HIDDEN / 8 + 4;  // 16-byte chunks of a row, shifted by 4 per token (bank conflicts)
    u32x4 y[few_tokens_most(HIDDEN)][kRow];      // normalised tokens
    f32x4 part[2][kFewWaves][64];                // the waves' shares of a tile, by the tile's parity
    float sums[kFewWaves][16];
};

// MULTI: the work-group has more than one chunk.
template <int HIDDEN, bool MULTI>
__device__ __forceinline__ void few_tokens_body(const FewTokensArgs& a, FewTokensLds<HIDDEN>& lds) {
    constexpr int kThreads = kFewWaves * 64;
    constexpr int STEPS = HIDDEN / (32 * kFewWaves);  // MFMA steps of a wave per tile
    constexpr int R = STEPS < 16 ? STEPS : 16;        // of a chunk
    constexpr int C = STEPS / R;                      // chunks per tile
    constexpr int TOKENS = few_tokens_most(HIDDEN);
    constexpr int PER = HIDDEN / 8 > kThreads ? HIDDEN / 8 / kThreads : 1;  // 16-byte chunks of a row per thread
    static_assert(STEPS * 32 * kFewWaves == HIDDEN && C * R == STEPS, "whole steps");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, quarter = lane >> 4;
    const int n_tokens = a.rope.n_tokens, D = a.rope.head_dim;
    const int nq = a.rope.n_q_heads * D, nkv = a.rope.n_kv_heads * D;
    const int n_tiles = (nq + 2 * nkv) / kTileOut;
    const int my_tiles = (n_tiles - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
    const bool norm = a.gamma != nullptr;

    // Where tile j of this work-group lies: matrix (Q, K, V) and first row of it.
    auto place = [&](int j, int* row0) {
        const int out0 = ((int)blockIdx.x + j * (int)gridDim.x) * kTileOut;
        const int which = out0 < nq ? 0 : out0 < nq + nkv ? 1 : 2;
        *row0 = out0 - (which == 0 ? 0 : which == 1 ? nq : nq + nkv);
        return which;
    };
    // Wave j finishes tile j; its lanes rotate pairs (row0 % D + 4 quarter) / 2 and the next of token `col`.
    int fin_row0 = 0, fin_which = 2;
    if (wave < my_tiles) fin_which = place(wave, &fin_row0);
    const bool rotate = a.rope.rope && fin_which < 2;
    float theta[2] = {};
    if (rotate) {
#pragma unroll
        for (int i = 0; i < 2; ++i) theta[i] = a.theta[((fin_row0 % D + 4 * quarter) >> 1) + i];
    }
    const u32x4* xr = reinterpret_cast<const u32x4*>(a.x);
    const bool in_row = HIDDEN / 8 >= kThreads || tid < HIDDEN / 8;
    u32x4 xv[TOKENS][PER], gv[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) gv[i] = norm && in_row ? reinterpret_cast<const u32x4*>(a.gamma)[i * kThreads + tid] : u32x4{};
#pragma unroll
    for (int t = 0; t < TOKENS; ++t)
        if (t < n_tokens) {
#pragma unroll
            for (int i = 0; i < PER; ++i) xv[t][i] = in_row ? xr[t * (HIDDEN / 8) + i * kThreads + tid] : u32x4{};
        }
    u32x4 w[2][R];  // chunks c and c + 1 of the work-group's stream of tiles
    const int n_chunks = my_tiles * C;
    auto load_w = [&](u32x4 (&dst)[R], int c) __attribute__((always_inline)) {
        int row0;
        const int which = place(c / C, &row0);
        const u32x4* wp = reinterpret_cast<const u32x4*>(a.w[which] + (size_t)(row0 + col) * HIDDEN +
                                                         wave * STEPS * 32 + (c % C) * R * 32 + 8 * quarter);
#pragma unroll
        for (int s = 0; s < R; ++s) dst[s] = __builtin_nontemporal_load(wp + 4 * s);
    };
    // Loads return in order, and a wait counts the ones behind it: the weights' loads are not conditional, so
    // that the wait for x leaves both chunks in flight, and the wait for a chunk the next one.
    load_w(w[0], 0);
    if constexpr (MULTI) load_w(w[1], 1);

    if (norm) {
#pragma unroll
        for (int t = 0; t < TOKENS; ++t)
            if (t < n_tokens) {
                float ss = 0.f;
#pragma unroll
                for (int i = 0; i < PER; ++i) {
                    ss += sum_squares(xv[t][i]);
                    asm volatile("" : "+v"(xv[t][i]));  // (the unpacked words are not kept for the scaling: registers)
                }
                ss = wave_sum(ss);
                if (lane == 0) lds.sums[wave][t] = ss;
            }
        __syncthreads();
        // (every lane: the scale of token `col`, handed out below)
        float total = 0.f;
#pragma unroll
        for (int i = 0; i < kFewWaves; ++i) total += lds.sums[i][col];
        const float inv = 1.0f / sqrtf(total / (float)HIDDEN + a.eps);
#pragma unroll
        for (int t = 0; t < TOKENS; ++t)
            if (t < n_tokens) {
                const float scale = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(inv), t));
#pragma unroll
                for (int i = 0; i < PER; ++i) xv[t][i] = scale_row(xv[t][i], gv[i], scale);
            }
    }
#pragma unroll
    for (int t = 0; t < TOKENS; ++t)
        if (t < n_tokens && in_row) {
#pragma unroll
            for (int i = 0; i < PER; ++i) lds.y[t][i * kThreads + tid] = xv[t][i];
        }
    float2 cs[2] = {};
    if (rotate) {
#pragma unroll
        for (int i = 0; i < 2; ++i) cs[i] = rope_cos_sin((fin_which == 0 ? a.q_pos_base : a.kv_pos_base) + col, theta[i]);
    }
    __syncthreads();

    const u32x4* yp = &lds.y[col < n_tokens ? col : 0][wave * STEPS * 4 + quarter];
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};  // output rows 4 quarter + i of the tile, token `col`
    auto product = [&](const u32x4 (&wc)[R], int c) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < R; ++s)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wc[s]),
                                                          __builtin_bit_cast(bf16x8_t, yp[((c % C) * R + s) * 4]), acc, 0, 0, 0);
    };
    auto finish = [&](int c) __attribute__((always_inline)) {  // after chunk c
        if (c % C != C - 1) return;
        const int j = c / C;
        lds.part[j & 1][wave][lane] = acc;
        acc = f32x4{0.f, 0.f, 0.f, 0.f};
        __syncthreads();  // (the other parity's readers have passed it, so its next writers may go on)
        if (wave != j || col >= n_tokens) return;
        f32x4 sum = lds.part[j & 1][0][lane];
#pragma unroll
        for (int i = 1; i < kFewWaves; ++i) sum += lds.part[j & 1][i][lane];
        uint32_t o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = f32_to_bf16_rne(sum[i]);
        uint2 out;
        out.x = rotate ? rotate_pair(o[0], o[1], cs[0].x, cs[0].y) : o[0] | (o[1] << 16);
        out.y = rotate ? rotate_pair(o[2], o[3], cs[1].x, cs[1].y) : o[2] | (o[3] << 16);
        const int head = fin_row0 / D;
        uint16_t* dst = fin_which == 0 ? a.rope.q_out + ((size_t)head * n_tokens + col) * D
                                       : cache_row(a.rope, fin_which == 1, head, col);
        if (dst != nullptr) *reinterpret_cast<uint2*>(dst + fin_row0 % D + 4 * quarter) = out;
    };
    if constexpr (!MULTI) {
        product(w[0], 0);
        finish(0);
    } else {
        int c = 0;
        for (; c + 3 < n_chunks; c += 2) {
            product(w[0], c);
            load_w(w[0], c + 2);
            finish(c);
            product(w[1], c + 1);
            load_w(w[1], c + 3);
            finish(c + 1);
        }
        if (c + 3 == n_chunks) {
            product(w[0], c);
            load_w(w[0], c + 2);
            finish(c);
            product(w[1], c + 1);
            finish(c + 1);
            product(w[0], c + 2);
            finish(c + 2);
        } else {
            product(w[0], c);
            finish(c);
            product(w[1], c + 1);
            finish(c + 1);
        }
    }
}

template <int HIDDEN>
__global__ __launch_bounds__(kFewWaves * 64) void layer_few_tokens_kernel(FewTokensArgs a) {
    __shared__ FewTokensLds<HIDDEN> lds;
    const int n_tiles = (a.rope.n_q_heads + 2 * a.rope.n_kv_heads) * a.rope.head_dim / kTileOut;
    constexpr bool kOneChunkTiles = HIDDEN <= 32 * kFewWaves * 16;
    if (kOneChunkTiles && (int)(blockIdx.x + gridDim.x) >= n_tiles)
        few_tokens_body<HIDDEN, !kOneChunkTiles>(a, lds);
    else
        few_tokens_body<HIDDEN, true>(a, lds);
}

}  // namespace

hipError_t launch_rms_norm(const NormArgs& args, const Launch& l) {
    NormArgs a = args;
    const int entries = a.table.cs ? a.table.sets * a.table.n_tokens * a.table.pairs : 0;
    a.table_wgs = (entries + kNormThreads - 1) / kNormThreads;
    const int rows = a.gamma ? a.n_tokens : 0;
    if (rows < 1 && a.table_wgs == 0) return hipSuccess;
    constexpr int rows_per_wg = kNormThreads / 64;
    const dim3 block(kNormThreads);
    if (rows > 0 && norm_vectorised(a)) {
        const dim3 grid(a.table_wgs + (rows + rows_per_wg - 1) / rows_per_wg);
        switch (a.hidden) {
            case 512: return launch_kernel(rms_norm_wave_kernel<1>, grid, block, l, a);
            case 1024: return launch_kernel(rms_norm_wave_kernel<2>, grid, block, l, a);
            case 2048: return launch_kernel(rms_norm_wave_kernel<4>, grid, block, l, a);
            case 4096: return launch_kernel(rms_norm_wave_kernel<8>, grid, block, l, a);
            case 8192: return launch_kernel(rms_norm_wave_kernel<16>, grid, block, l, a);
            default: break;
        }
    }
    return launch_kernel(rms_norm_kernel, dim3(a.table_wgs + rows), block, l, a);
}

hipError_t launch_rope_scatter(const RopeArgs& a, const Launch& l) {
    if (a.n_tokens < 1) return hipSuccess;
    if (a.head_dim < 8 || a.head_dim > 2 * kMaxRopePairs || (a.head_dim & 7) || kRopeThreads % (a.head_dim / 8) ||
        (a.rope && a.cs == nullptr))
        return hipErrorInvalidValue;
    return launch_kernel(rope_scatter_kernel, dim3(a.n_tokens), dim3(kRopeThreads), l, a);
}

static int few_tokens_tiles(const FewTokensArgs& a) {
    return (a.rope.n_q_heads + 2 * a.rope.n_kv_heads) * a.rope.head_dim / kTileOut;
}

bool few_tokens_supported(const FewTokensArgs& a, int n_cu) {
    const uintptr_t align = reinterpret_cast<uintptr_t>(a.x) | reinterpret_cast<uintptr_t>(a.gamma) |
                            reinterpret_cast<uintptr_t>(a.w[0]) | reinterpret_cast<uintptr_t>(a.w[1]) |
                            reinterpret_cast<uintptr_t>(a.w[2]);
    return a.rope.n_tokens >= 1 && a.rope.n_tokens <= few_tokens_most(a.hidden) && a.rope.head_dim % kTileOut == 0 &&
           (align & 15) == 0 && few_tokens_tiles(a) <= kFewWaves * n_cu &&
           (a.hidden == 1024 || a.hidden == 2048 || a.hidden == 4096 || a.hidden == 8192);
}

hipError_t launch_few_tokens(const FewTokensArgs& a, int n_cu, const Launch& l) {
    if (!few_tokens_supported(a, n_cu)) return hipErrorInvalidValue;
    const dim3 grid(std::min(few_tokens_tiles(a), n_cu));
    const dim3 block(kFewWaves * 64);
    switch (a.hidden) {
        case 1024: return launch_kernel(layer_few_tokens_kernel<1024>, grid, block, l, a);
        case 2048: return launch_kernel(layer_few_tokens_kernel<2048>, grid, block, l, a);
        case 4096: return launch_kernel(layer_few_tokens_kernel<4096>, grid, block, l, a);
        default: return launch_kernel(layer_few_tokens_kernel<8192>, grid, block, l, a);
    }
}

}  // namespace lara
