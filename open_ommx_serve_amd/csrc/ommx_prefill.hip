// Causal attention of prompt rows over their own bf16 K/V: the read side of a full-prefill step (the
// reference leaves it to the engine's varlen kernel, ommx_gpu_serve/integration/vllm/backend.py).
// Grouped-query heads, any number of requests per launch, head_dim 64 or 128.
//
// Precision is that of an fp32 softmax: q.k of bf16 operands is exact in the fp32 accumulator, the weights
// p = exp2(s - m) are fp32 and enter P.V times 2^8 as two f16 pieces (11 bits, then the remainder rounded to 11) against
// V times 2^8 in f16, which is exact for every bf16 of magnitude 2^-22 to 256 and zero.  Two pieces hold a weight to
// 2^-23 of itself down to 2^-10 of the row's largest, and to 2^-33 of the largest below.  A 64-key tile with any other
// V element is left out of the loop and follows in a second pass, with the weights in three bf16 pieces (all 24 bits)
// and V as it is.  The second pass also takes every tile where the small weights of some row are all that counts (its
// largest ones met a V of next to nothing: an attention sink), which the sums at the end of the loop show; both passes
// together take 2.1 times as long.  Relative error against fp64, and that of the library's fp32 attention: 4096 rows
// with K outliers 7.0e-7 and 1.2e-6; 4096, 700 and 100 plain rows 2.9e-7, 1.9e-7, 1.4e-7 and 4.8e-7, 2.5e-7, 1.5e-7;
// one key of V = 0 that outweighs every other 2^16 or 2^24 times 7.2e-7, 8.9e-7 and 1.1e-6, 1.4e-6 (without the second
// pass and at 2^6 instead of 2^8 6.6e-6, 1.6e-3).
//
// Layout.  A group of four waves = 128 query rows of one q head; a wave owns 32 rows and walks the keys
// 64 at a time with mfma_f32_32x32x16.  Scores are formed transposed, S^T = K.Q^T, so a lane
// holds 32 scores of ONE query row: maximum and sum are register work plus one exchange with the
// other half of the wave.  The accumulator rows a lane holds (8j + 4*half + 0..3) are, in this order, what
// the B operand of O^T = V^T.P^T wants for a 16-key block once V^T lists its keys in the same order,
// so the weights never pass through LDS.  K rows and transposed V are double buffered in LDS (70 KB); the next tile's
// rows are requested before a tile is worked on, through buffers that end with the request.
//
// Bound: power, once the chip is full.  4096 tokens of 32 heads: 203 K clocks of matrix instructions and 203 K of vector
// ones in 363 K (rocprofv3 counters), and those pass at 1.8 GHz: a tile step of a workgroup takes 3.03 us with 512 of
// them and 1.93 us with 128 (8 heads), both alone on their compute units, and 1.05 PFLOP/s issued compares with 1.21 of a
// large library product on the same card.  The two kinds of instructions hardly hold each other up (a vector instruction
// 7.45 clocks beside a wave of matrix instructions, 6.8 without; the matrix ones the same), and dealing the staging out
// evenly over both groups of waves changed nothing (206.7 -> 212.5 us).  That is
// 191 to 200 us from card to card (HIP events around launches back to back; the kernel trace of rocprofv3 has 204 at least
// and 207 on average).  Two groups of waves in one workgroup, one half a tile behind the other so that the matrix phase of
// one meets the vector phase of the other, share the staged tiles as well: 264 -> 191 us (events, one card, with two pieces
// and no second pass).  In lockstep, without the shift, the eight waves took 210 us, as two workgroups of four 233 us; any
// register spilled in the loop costs more than all of this, because its reload waits for the loads on their way (285 us).
// Short prompts are latency: one group per workgroup, two workgroups per compute unit (see prefill_attention).  Where the
// workgroups leave compute units idle beside the longest chain of tiles, two groups take the keys of the same rows, every
// other tile each with staging of its own and half a tile apart, and their sums are put together through LDS (SPLIT): 1.4 us a
// tile of the chain instead of 2.1.  In lockstep, without the shift, 1024 rows took 39.0 us instead of 36.3 (one group 42.5).  The
// library's fp32 attention took 2.45 ms.
#include <algorithm>

#include "ommx_common.h"
#include "ommx_internal.h"

namespace ommx {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

struct PrefillArgs {
    const uint16_t *q, *k, *v;
    int64_t q_t, q_h, k_t, k_h, v_t, v_h;
    float* o;
    uint16_t* o16;
    int64_t o_t, o_h;
    int Hkv, R;
    float scale_log2;            // softmax scale times log2(e)
};

constexpr int QROWS = 128, KEYS = 64;
// {first row of the request, its length, first query row of the tile within it}
constexpr int kTilesPerLaunch = kUploadWords / 3;
struct TileList { int32_t w[kUploadWords]; };

__device__ __forceinline__ f32x16 mfma_bf16(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma_f16(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ float other_half(float v) { return __shfl_xor(v, 32); }
// high halves of two words: elements 0 and 1 of a packed bf16 pair, truncated
__device__ __forceinline__ uint32_t hi_pair(float lo, float hi) {
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}
// x less one half of a packed f16 pair, one instruction (the compiler converts first)
__device__ __forceinline__ float minus_low(float x, f16x2 h) {
    float r;
    asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(x));
    return r;
}
__device__ __forceinline__ float minus_high(float x, f16x2 h) {
    float r;
    asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(x));
    return r;
}
__device__ __forceinline__ u32x4 load16(__amdgpu_buffer_rsrc_t rows, uint32_t at) {
    return __builtin_amdgcn_raw_buffer_load_b128(rows, at, 0, 0);
}

// The running maximum is refreshed when a score (base 2) exceeds it by the slack: any bound that keeps
// exp2 in range serves an online softmax, and most tiles then rescale nothing.
// Weights are carried times 2^8, at most 2^15.75 with the slack, within f16.  More would leave less to the second pass,
// but the shift is part of exp2's argument, which is rounded to 24 bits: at 2^9 and above plain short rows are less exact
// than the library's (1.6e-7, at 2^12 2.0e-7, against 1.5e-7), and the smaller slack rescales more tiles (4096 rows, at
// 2^8 and 2^12: 2 % and 3.5 % above 2^6 without the second pass).  The gain as a factor of its own costs 5 to 7 % (plain
// multiplications, mixed-precision fused ones).
// V is carried times 2^8 and divided by it at the end.
constexpr float P_SHIFT = 8.0f, MAX_SLACK = 7.75f, V_GAIN = 256.0f;
// In the second pass the sums so far and its weights are carried times this: a V of 2^100 is still in range.
constexpr float LATE_GAIN = 1.0f / 16384;
// Rows whose largest sum is below this times sqrt(n) times the largest V go through the second pass.  The pieces are off
// by 2^-25 at most, 2^-25.8 on average, so n of them leave sqrt(n) * 2^-25.8 of a V of average size, about a quarter of the
// largest, in a sum about a third of the row's largest: 2^-21.3 of it at the line.
constexpr float AGAIN_BELOW = 1.0f / 32;
// a bf16 value times 2^8 is exactly an f16 when its magnitude bits are 0 or in this range (2^-22 to 256)
constexpr unsigned short V_LOW = (104 + 1) << 7, V_HIGH = ((104 + 31) << 7) - 1;

// LDS rows are 16 bytes longer than their data: eight neighbouring rows start in different bank groups, and every
// operand read is one lane address plus an immediate offset (an XOR swizzle kept 36 addresses in registers)
constexpr int k_stride(int D) { return 2 * D + 16; }
constexpr int V_STRIDE = 2 * KEYS + 16;

// GROUPS 2: two groups of waves that share the staged tiles.  SPLIT: two that take the even and the odd tiles of the same rows.
template <int D, int GROUPS, bool SPLIT = false>
__global__ void __launch_bounds__(SPLIT ? 512 : 256 * GROUPS, 2) prefill_kernel(PrefillArgs a, TileList tiles) {
    constexpr int KB = D / 16;           // 16-channel blocks of QK
    constexpr int DB = D / 32;           // 32-channel blocks of the output
    constexpr int CHUNKS = D / 8;        // 16-byte chunks of a K row
    constexpr int KS = k_stride(D), VS = V_STRIDE;
    constexpr int KLOADS = KEYS * CHUNKS / 256;
    static_assert(!SPLIT || GROUPS == 1, "groups that split the keys stage for themselves, as one group does");
    constexpr int STEP = SPLIT ? 2 : 1;              // tiles from one of a group's to its next
    constexpr int K_BUF = KEYS * KS, V_BUF = D * VS, GROUP_LDS = 2 * (K_BUF + V_BUF);
    __shared__ __attribute__((aligned(16))) uint8_t s_kv[STEP][GROUP_LDS];       // K rows and transposed V, two tiles each
    __shared__ uint32_t s_inexact[kPrefillMaxRows / KEYS / 32];          // bit per tile: some V element is no f16
    __shared__ uint32_t s_top, s_again;              // largest |V| of the other tiles; a row wants all tiles again
    __shared__ int s_first[3][D], s_special;         // first row with +inf, -inf, NaN in a channel of V; whether there is one
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, half = lane >> 5, group = GROUPS == 2 || SPLIT ? wave >> 2 : 0;
    uint8_t* const lds = s_kv[SPLIT ? group : 0];
    auto s_k = [&](int t) { return lds + (t / STEP & 1) * K_BUF; };
    auto s_v = [&](int t) { return lds + 2 * K_BUF + (t / STEP & 1) * V_BUF; };
    const int t0 = tiles.w[3 * blockIdx.y], len = tiles.w[3 * blockIdx.y + 1], q0 = tiles.w[3 * blockIdx.y + 2];
    // (neighbouring workgroups take neighbouring kv heads, so with 8 kv heads an XCD keeps to one)
    const int kvh = blockIdx.x % a.Hkv, part = blockIdx.x / a.Hkv;
    const bool pair = GROUPS == 2 && a.R % 2 == 0;          // the groups take two q heads, else two row blocks of one
    const int h = kvh * a.R + (pair ? 2 * part + group : part);
    const uint16_t* const kp = a.k + t0 * a.k_t + kvh * a.k_h;
    const uint16_t* const vp = a.v + t0 * a.v_t + kvh * a.v_h;

    const int row_first = q0 + 32 * (wave & 3) + (pair || SPLIT ? 0 : QROWS * group), row = row_first + col;   // of this wave, of this lane
    u32x4 qf[KB];
    {
        const uint16_t* qp = a.q + (t0 + min(row, len - 1)) * a.q_t + h * a.q_h + 8 * half;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) qf[kb] = *reinterpret_cast<const u32x4*>(qp + 16 * kb);
    }
    f32x16 acc[DB];
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[d][r] = 0.0f;
    float m = -INFINITY, l = 0.0f;       // m: running maximum less P_SHIFT

    // key tiles of the workgroup and of this wave (causal; a wave whose rows are past the end has none)
    const int n_tiles = (min(len, q0 + (pair ? QROWS : GROUPS * QROWS)) + KEYS - 1) / KEYS;
    int n_mine = row_first < len ? min(n_tiles, (row_first + 31) / KEYS + 1) : 0;

    // ---- staging.  The first group brings V: channels 8*d8.. of four neighbouring rows per thread, sixteen lanes write a
    // whole row of transposed V (head_dim 64: half of the threads).  The second group brings K: chunk kc of rows kr, ...
    const int st = tid & 255;
    const int kc = st % CHUNKS, kr = st / CHUNKS;
    const int kg = st % (KEYS / 4), d8 = st / (KEYS / 4);
    const uint32_t k_row = static_cast<uint32_t>(a.k_t) * 2, v_row = static_cast<uint32_t>(a.v_t) * 2;
    const uint32_t k_at = kr * k_row + 16 * kc, v_at = 4 * kg * v_row + 16 * d8;
    u16x2 v_top = {0, 0};                // largest |V| this thread has staged
    u32x4 nx[GROUPS == 2 ? 4 : 8];       // rows on their way: V, K behind it (two groups: either)
    u32x4* const nk = nx + (GROUPS == 2 ? 0 : 4);
    // The rows of a tile as a buffer that ends with the request's last row: loads beyond it return zeros.
    auto tile_rows = [&](const uint16_t* p, int64_t stride, int t) {
        const int rows = min(len - t * KEYS, KEYS);
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p + t * KEYS * stride), 0,
                                                 (rows - 1) * static_cast<int>(stride) * 2 + 2 * D, 0x00027000);
    };
    auto request_k = [&](int t) {
        if (t >= n_tiles) return;
        const auto rows = tile_rows(kp, a.k_t, t);
#pragma unroll
        for (int i = 0; i < KLOADS; ++i) nk[i] = load16(rows, k_at + i * (256 / CHUNKS) * k_row);
    };
    auto request_v = [&](int t) {
        if (t >= n_tiles || d8 >= CHUNKS) return;
        const auto rows = tile_rows(vp, a.v_t, t);
#pragma unroll
        for (int i = 0; i < 4; ++i) nx[i] = load16(rows, v_at + i * v_row);
    };
    auto write_v = [&](int t, const u32x4* f) {
        // keys 4kg..4kg+3 are block kg / 4, half kg & 1 of it, first or second four slots of that chunk
        uint8_t* const at = s_v(t) + 8 * d8 * VS + 16 * (2 * (kg >> 2) + (kg & 1)) + 8 * ((kg >> 1) & 1);
#pragma unroll
        for (int w = 0; w < 4; ++w)
#pragma unroll
            for (int odd = 0; odd < 2; ++odd) {
                const uint32_t sel = odd ? 0x07060302u : 0x05040100u;
                *reinterpret_cast<u32x2*>(at + (2 * w + odd) * VS) =
                    u32x2{__builtin_amdgcn_perm(f[1][w], f[0][w], sel), __builtin_amdgcn_perm(f[3][w], f[2][w], sel)};
            }
    };
    auto stage_k = [&](int t) {
        if (t >= n_tiles) return;
#pragma unroll
        for (int i = 0; i < KLOADS; ++i)
            *reinterpret_cast<u32x4*>(s_k(t) + (kr + i * (256 / CHUNKS)) * KS + 16 * kc) = nk[i];
    };
    auto stage_v = [&](int t) {
        if (d8 >= CHUNKS) return;
        // V * 2^8 as f16: the exponent field shifted down by 104, three more mantissa bits; zero stays zero
        u16x2 low = {0xFFFF, 0xFFFF}, high = {0, 0};
        u32x4 f[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const uint32_t x = nx[i][w];
                const u16x2 mag = __builtin_bit_cast(u16x2, x & 0x7FFF7FFFu);
                low = __builtin_elementwise_min(low, mag - static_cast<unsigned short>(1));      // zero wraps to the top
                high = __builtin_elementwise_max(high, mag);
                const u16x2 bias = {104 << 7, 104 << 7};
                f[i][w] = (x & 0x80008000u) | __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(mag, bias) << 3);
            }
        if (min(low[0], low[1]) < V_LOW - 1 || max(high[0], high[1]) > V_HIGH) atomicOr(&s_inexact[t >> 5], 1u << (t & 31));
        else v_top = __builtin_elementwise_max(v_top, high);
        write_v(t, f);
    };
    // Elements of V that are no number are taken out of the staged rows, where a weight of zero (a row before them, a
    // piece of a weight) would turn them into NaN, and noted: every row from theirs on gets them in the end.
    auto take_special = [&](int t) {
        u16x2 high = {0, 0};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int w = 0; w < 4; ++w) high = __builtin_elementwise_max(high, __builtin_bit_cast(u16x2, nx[i][w] & 0x7FFF7FFFu));
        if (max(high[0], high[1]) < 0x7F80) return;
        s_special = 1;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t x = nx[i][e >> 1] >> (16 * (e & 1)) & 0xFFFFu;
                if ((x & 0x7FFFu) < 0x7F80u) continue;
                atomicMin(&s_first[x == 0x7F80u ? 0 : (x == 0xFF80u ? 1 : 2)][8 * d8 + e], t * KEYS + 4 * kg + i);
                nx[i][e >> 1] &= e & 1 ? 0x0000FFFFu : 0xFFFF0000u;
            }
    };
    auto inexact = [&](int t) { return (__builtin_amdgcn_readfirstlane(s_inexact[t >> 5]) >> (t & 31)) & 1u; };

    f32x16 s[2];                 // scores of the tile, transposed: lane's row is the query
    u32x4 p0[4], p1[4];          // their weights in two f16 pieces, by 16-key block

    auto v_operand = [&](int t, int b, int d) {
        return *reinterpret_cast<const u32x4*>(s_v(t) + (32 * d + col) * VS + 32 * b + 16 * half);
    };
    auto scores = [&](int t) {
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[g][r] = 0.0f;
        u32x4 kf[2][2][2];
        auto read = [&](int kb2) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                kf[kb2 & 1][i >> 1][i & 1] =
                    *reinterpret_cast<const u32x4*>(s_k(t) + (32 * (i & 1) + col) * KS + 32 * (2 * kb2 + (i >> 1)) + 16 * half);
        };
        read(0);
#pragma unroll
        for (int kb2 = 0; kb2 < KB / 2; ++kb2) {
            if (kb2 + 1 < KB / 2) read(kb2 + 1);
#pragma unroll
            for (int i = 0; i < 4; ++i) s[i & 1] = mfma_bf16(kf[kb2 & 1][i >> 1][i & 1], qf[2 * kb2 + (i >> 1)], s[i & 1]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto mask = [&](int t) {
        const int k0 = t * KEYS;
        if (k0 + KEYS - 1 <= row_first) return;
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (k0 + 32 * g + 8 * (r >> 2) + 4 * half + (r & 3) > row) s[g][r] = -INFINITY;
    };
    // O^T += V^T.P^T of one tile
    auto add_pv = [&](int t) {
        if (inexact(t)) return;              // (follows after the loop)
        u32x4 vf[2][DB];                     // operands one block ahead, no further: registers
#pragma unroll
        for (int d = 0; d < DB; ++d) vf[0][d] = v_operand(t, 0, d);
#pragma unroll
        for (int b = 0; b < 4; ++b) {
#pragma unroll
            for (int d = 0; d < DB; ++d)
                if (b < 3) vf[(b + 1) & 1][d] = v_operand(t, b + 1, d);
#pragma unroll
            for (int d = 0; d < DB; ++d) acc[d] = mfma_f16(vf[b & 1][d], p0[b], acc[d]);
#pragma unroll
            for (int d = 0; d < DB; ++d) acc[d] = mfma_f16(vf[b & 1][d], p1[b], acc[d]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // a row none of whose keys in this group has had any weight so far (scores of -inf): SPLIT, where the first tile is not every row's
    auto finite = [](float x) { return SPLIT && x == -INFINITY ? 0.0f : x; };
    // vector phase: staging, then the online softmax of one row per lane
    auto vector_phase = [&](int t) {
        if (GROUPS == 1 || !group) {
            if (!SPLIT || t < n_tiles) stage_v(t);
            request_v(t + STEP);
        }
        if (GROUPS == 1) { stage_k(t + STEP); request_k(t + 2 * STEP); }
        else if (group) { stage_k(t + 2); request_k(t + 3); }
        if (SPLIT && t >= n_mine) return;        // (all keys masked: there may be no maximum yet)
        mask(t);
        float mx = s[0][0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[0][r]);
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[1][r]);
        mx = fmaf(fmaxf(mx, other_half(mx)), a.scale_log2, -P_SHIFT);      // (the scale is positive)
        if (__any(mx > m + MAX_SLACK)) {
            const float m_new = fmaxf(m, mx);
            const float shrink = __builtin_amdgcn_exp2f(m - finite(m_new));       // 0 on the first tile
            m = m_new;
            l *= shrink;
#pragma unroll
            for (int d = 0; d < DB; ++d)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[d][r] *= shrink;
        }
        const float less = finite(m);
        float tile_l = 0.0f;      // (of its own: next to a large weight small ones would be rounded off one by one)
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float x = __builtin_amdgcn_exp2f(fmaf(s[b >> 1][8 * (b & 1) + 2 * i], a.scale_log2, -less));
                const float y = __builtin_amdgcn_exp2f(fmaf(s[b >> 1][8 * (b & 1) + 2 * i + 1], a.scale_log2, -less));
                tile_l += x + y;
                const f16x2 hi = __builtin_convertvector((f32x2{x, y}), f16x2);
                const f32x2 rest = {minus_low(x, hi), minus_high(y, hi)};
                p0[b][i] = __builtin_bit_cast(uint32_t, hi);
                p1[b][i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(rest, f16x2));
            }
        l += tile_l;
        if (GROUPS == 2 || SPLIT) {        // all of it here: the compiler would move the weights behind the barrier, to their use
#pragma unroll
            for (int b = 0; b < 4; ++b) asm volatile("" : "+v"(p0[b]), "+v"(p1[b]));
            asm volatile("" : "+v"(l));
        }
    };

    if (tid < kPrefillMaxRows / KEYS / 32) s_inexact[tid] = 0;
    if (tid < D) s_first[0][tid] = s_first[1][tid] = s_first[2][tid] = INT32_MAX;
    if (tid == 0) s_top = s_again = s_special = 0;
    const int t_first = SPLIT ? group : 0;
    if (GROUPS == 1 || group) { request_k(t_first); stage_k(t_first); request_k(t_first + STEP); }
    if (GROUPS == 1 || !group) request_v(t_first);
    __syncthreads();
    if (group) {                  // one phase behind the first group
        if (GROUPS == 2) { stage_k(1); request_k(2); }
        __syncthreads();
    }
    if (!SPLIT || t_first < n_mine) scores(t_first);
    if (GROUPS == 2 || SPLIT) __syncthreads();
    for (int t0s = 0; t0s < n_tiles; t0s += STEP) {
        const int t = t0s + t_first;
        vector_phase(t);
        __syncthreads();
        if (!SPLIT || t < n_mine) add_pv(t);
        if (t + STEP < (SPLIT ? n_mine : n_tiles)) scores(t + STEP);
        else asm volatile("" : "=v"(s[0]), "=v"(s[1]));           // (keeps the scores out of the loop's registers)
        if ((GROUPS == 2 || SPLIT) && (!group || t0s + STEP < n_tiles)) __syncthreads();
    }
    if constexpr (SPLIT) {
        // the second group's sums to the first, which goes on alone (the second keeps its barriers company)
        static_assert(GROUP_LDS >= (4 * DB + 1) * 256 * 16, "sums of a group");
        f32x4* const there = reinterpret_cast<f32x4*>(s_kv[1]) + st;
        __syncthreads();
        if (group) {
#pragma unroll
            for (int i = 0; i < 4 * DB; ++i)
                there[256 * i] = f32x4{acc[i >> 2][4 * (i & 3)], acc[i >> 2][4 * (i & 3) + 1], acc[i >> 2][4 * (i & 3) + 2], acc[i >> 2][4 * (i & 3) + 3]};
            there[256 * 4 * DB] = f32x4{m, l, 0.0f, 0.0f};
            n_mine = 0;
        }
        __syncthreads();
        if (!group && n_mine > 0) {
            const f32x4 ml = there[256 * 4 * DB];
            const float m_new = fmaxf(m, ml[0]);
            const float mine = __builtin_amdgcn_exp2f(m - m_new), other = __builtin_amdgcn_exp2f(ml[0] - m_new);
            m = m_new;
            l = l * mine + ml[1] * other;
#pragma unroll
            for (int i = 0; i < 4 * DB; ++i) {
                const f32x4 x = there[256 * i];
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i >> 2][4 * (i & 3) + r] = acc[i >> 2][4 * (i & 3) + r] * mine + x[r] * other;
            }
        }
    }

    // Second pass over tiles whose V is not exact in f16: scores once more, weights against the final maximum in three bf16
    // pieces (8 + 8 + 8 bits by truncation, their sum is the weight), V as it is.
    float gain = V_GAIN;
    auto second_pass = [&](auto tiles_of, float keep) {
        bool first = true;
        for (int w = 0; w <= (n_tiles - 1) >> 5; ++w)
            for (uint32_t left = tiles_of(w); left; left &= left - 1) {
                const int t = 32 * w + __builtin_ctz(left);
                if (SPLIT ? !group : GROUPS == 1 || group) {
                    request_k(t);
                    stage_k(t);
                }
                if ((SPLIT ? !group : GROUPS == 1 || !group) && d8 < CHUNKS) {
                    request_v(t);
                    take_special(t);
                    write_v(t, nx);
                }
                if (first) {
#pragma unroll
                    for (int d = 0; d < DB; ++d)
#pragma unroll
                        for (int r = 0; r < 16; ++r) acc[d][r] *= keep;
                    gain = V_GAIN * LATE_GAIN;
                    first = false;
                }
                __syncthreads();
                if (t < n_mine) {
                    scores(t);
                    mask(t);
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        float x[8];
#pragma unroll
                        for (int i = 0; i < 8; ++i)
                            x[i] = __builtin_amdgcn_exp2f(fmaf(s[b >> 1][8 * (b & 1) + i], a.scale_log2, -m)) * (V_GAIN * LATE_GAIN);
#pragma unroll
                        for (int n = 0; n < 3; ++n) {
                            u32x4 p;
#pragma unroll
                            for (int i = 0; i < 4; ++i) p[i] = hi_pair(x[2 * i], x[2 * i + 1]);
#pragma unroll
                            for (int i = 0; i < 8; ++i) x[i] -= __uint_as_float(__float_as_uint(x[i]) & 0xFFFF0000u);
#pragma unroll
                            for (int d = 0; d < DB; ++d) acc[d] = mfma_bf16(v_operand(t, b, d), p, acc[d]);
                        }
                    }
                }
                __syncthreads();
            }
    };
    for (int i = 32; i; i >>= 1)
        v_top = __builtin_elementwise_max(v_top, __builtin_bit_cast(u16x2, __shfl_xor(__builtin_bit_cast(int, v_top), i)));
    if (lane == 0) atomicMax(&s_top, static_cast<uint32_t>(max(v_top[0], v_top[1])));
    __syncthreads();
    second_pass([&](int w) -> uint32_t { return __builtin_amdgcn_readfirstlane(s_inexact[w]); }, LATE_GAIN);

    // Rows whose sums are small against V: see AGAIN_BELOW.
    {
        float most = 0.0f;
#pragma unroll
        for (int d = 0; d < DB; ++d)
#pragma unroll
            for (int r = 0; r < 16; ++r) most = fmaxf(most, fabsf(acc[d][r]));
        most = fmaxf(most, other_half(most));
        const float top = __uint_as_float(s_top << 16) * gain * AGAIN_BELOW;
        if (row < len && !(SPLIT && group) && most * most < top * top * static_cast<float>(row + 1)) s_again = 1;
    }
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(s_again))
        second_pass([&](int w) { return n_tiles - 32 * w >= 32 ? ~0u : (1u << (n_tiles - 32 * w)) - 1; }, 0.0f);

    const bool special = __builtin_amdgcn_readfirstlane(s_special);
    if (row >= len || (SPLIT && group)) return;
    l += other_half(l);
    const float inv = 1.0f / (l * gain);
    const int64_t at = (t0 + row) * a.o_t + h * a.o_h;
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            const int ch = 32 * d + 8 * r4 + 4 * half;
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = acc[d][4 * r4 + i] * inv;
            if (special)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (row >= s_first[0][ch + i]) v[i] += INFINITY;
                    if (row >= s_first[1][ch + i]) v[i] -= INFINITY;
                    if (row >= s_first[2][ch + i]) v[i] = NAN;
                }
            if (a.o16)
                *reinterpret_cast<u32x2*>(a.o16 + at + ch) =
                    u32x2{f32_to_bf16_any(v[0]) | (static_cast<uint32_t>(f32_to_bf16_any(v[1])) << 16),
                          f32_to_bf16_any(v[2]) | (static_cast<uint32_t>(f32_to_bf16_any(v[3])) << 16)};
            else
                *reinterpret_cast<float4*>(a.o + at + ch) = float4{v[0], v[1], v[2], v[3]};
        }
}

template <int D>
void launch(const PrefillArgs& a, const TileList& list, int n, PrefillForm form, hipStream_t st) {
    if (form == PrefillForm::two_groups)
        hipLaunchKernelGGL((prefill_kernel<D, 2>), dim3(a.R % 2 ? a.Hkv * a.R : a.Hkv * a.R / 2, n), dim3(512), 0, st, a, list);
    else if (form == PrefillForm::split_keys)
        hipLaunchKernelGGL((prefill_kernel<D, 1, true>), dim3(a.Hkv * a.R, n), dim3(512), 0, st, a, list);
    else
        hipLaunchKernelGGL((prefill_kernel<D, 1>), dim3(a.Hkv * a.R, n), dim3(256), 0, st, a, list);
}

}  // namespace

// Two wave groups per workgroup pay when the tiles are long and fill the chip: they halve the vector work of staging
// and overlap matrix and vector work, but a workgroup is twice as large and runs half a tile longer.  One group -> two
// groups, us, 32 q / 8 kv heads: 4096 rows 246 -> 208, 2048 80.5 -> 79.3, 8 x 1024 141 -> 137; 1024 38.5 -> 42.1
// (half the chip), 16 x 512 95 -> 126 (five key tiles a workgroup on average), 100 rows 9.8 -> 13.0.
// One group a workgroup leaves compute units idle, or half empty, while the longest tiles are at their keys: then those are
// split.  Kernel alone, one group -> split, us, 32 q / 8 kv heads: 100 rows 11.8 -> 13.4, 200 15.4 -> 15.5, 300 17.6 -> 16.9, 433 21.7 ->
// 20.0, 622 29.7 -> 26.0, 1024 42.5 -> 36.3, head_dim 64 35.5 -> 30.6; 4000 rows of 8 heads 131.8 -> 99.7.
// A compute unit holds one workgroup with its keys split, two of one group.  Two rounds of the former pay where what a compute
// unit has to do in all, key_tiles * Hq / 256 tiles, is little beside the longest chain: 1100 rows (18 tiles, 11 a unit) 46.5 ->
// 36.4, 1900 (30, 30) 73.1 -> 64.0, beside short prompts 1100 + 7 x 100 (13) 43.8 -> 41.4, 1100 + 600 (15) 44.5 -> 41.0, 1500 + 3 x 128 (24, 20)
// 57.7 -> 53.3, 4000 + 30 x 100 of 8 heads 122.9 -> 89.6; equal prompts of 8 heads 6 x 1100 (16.9) 45.2 -> 44.3, 5 x 1500 (24, 24.4) 59.0 ->
// 55.5, but 7 x 1030 (17, 19.5) 44.5 -> 47.6, head_dim 64 34.4 -> 40.6, 6 x 1200 (19, 20.4) 47.3 -> 48.9 and 38.0 -> 41.0; shorter chains 2 x 768 37.8 -> 38.8,
// 3 x 512 29.6 -> 35.0, 8 x 256 24.8 -> 35.9.  The line lies where the two meet over 122 batches of 17 tiles and more, 4 to 32
// heads (at head_dim 64 tiles are shorter beside what a workgroup does once): the other form would be better by 2.7 % for one of
// them, by at most 1.4 % for the rest.
PrefillForm prefill_form(const int64_t* host_starts, int B, int Hq, int D) {
    int64_t groups = 0, key_tiles = 0, longest = 0;
    for (int b = 0; b < B; ++b)
        for (int64_t q0 = 0, len = host_starts[b + 1] - host_starts[b]; q0 < len; q0 += QROWS) {
            const int64_t keys = (std::min<int64_t>(len, q0 + QROWS) + KEYS - 1) / KEYS;
            ++groups;
            key_tiles += keys;
            longest = std::max(longest, keys);
        }
    const int64_t workgroups = groups * Hq;
    if (workgroups >= 2 * 256 && key_tiles >= 8 * groups) return PrefillForm::two_groups;
    if (workgroups <= 256) return longest >= 5 ? PrefillForm::split_keys : PrefillForm::one_group;
    const bool two_rounds = workgroups <= 2 * 256 && longest > 16 && 2 * key_tiles * Hq <= 256 * (3 * longest - (D == 128 ? 18 : 20));
    return two_rounds ? PrefillForm::split_keys : PrefillForm::one_group;
}

int prefill_attention(const uint16_t* q, int64_t q_t, int64_t q_h, const uint16_t* k, int64_t k_t, int64_t k_h,
                      const uint16_t* v, int64_t v_t, int64_t v_h, void* o, bool o_bf16, int64_t o_t, int64_t o_h,
                      const int64_t* host_starts, int B, int Hq, int Hkv, int D, float scale, void* stream) {
    const char* bad = nullptr;
    if (B < 1 || Hkv < 1 || Hq % Hkv || !(D == 64 || D == 128) || !(scale > 0.0f)) bad = "prefill_attention: bad shape";
    else if (((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) |
               reinterpret_cast<uintptr_t>(o)) & 15) ||
             (q_t | q_h | k_t | k_h | v_t | v_h | o_t | o_h) % 8)
        bad = "prefill_attention: rows must be 16-byte aligned";
    else if (k_t >= kPrefillMaxStride || v_t >= kPrefillMaxStride) bad = "prefill_attention: K / V rows too far apart";
    for (int b = 0; b < B && !bad; ++b)
        if (host_starts[b + 1] - host_starts[b] > kPrefillMaxRows) bad = "prefill_attention: request too long";
    if (bad) { set_error(bad); return -1; }
    const PrefillArgs a{q, k, v, q_t, q_h, k_t, k_h, v_t, v_h, o_bf16 ? nullptr : static_cast<float*>(o),
                        o_bf16 ? static_cast<uint16_t*>(o) : nullptr, o_t, o_h, Hkv, Hq / Hkv,
                        scale * 1.4426950408889634f};
    // Tiles of 128 query rows, those with the most keys first: the grid drains evenly.
    int most = 0;
    for (int b = 0; b < B; ++b) {
        const int64_t n = host_starts[b + 1] - host_starts[b];
        if (n > most) most = static_cast<int>(n);
    }
    const PrefillForm form = prefill_form(host_starts, B, Hq, D);
    TileList list;
    int n = 0;
    hipStream_t st = static_cast<hipStream_t>(stream);
    auto flush = [&]() {
        if (n == 0) return;
        if (D == 128) launch<128>(a, list, n, form, st); else launch<64>(a, list, n, form, st);
        n = 0;
    };
    const int step = form == PrefillForm::two_groups && a.R % 2 ? 2 * QROWS : QROWS;
    for (int q0 = (most - 1) / step * step; q0 >= 0; q0 -= step)
        for (int b = 0; b < B; ++b) {
            const int len = static_cast<int>(host_starts[b + 1] - host_starts[b]);
            if (q0 >= len) continue;
            list.w[3 * n] = static_cast<int32_t>(host_starts[b]);
            list.w[3 * n + 1] = len;
            list.w[3 * n + 2] = q0;
            if (++n == kTilesPerLaunch) flush();
        }
    flush();
    if (hipGetLastError() != hipSuccess) { set_error("prefill_attention: launch failed"); return -2; }
    return 0;
}

}  // namespace ommx
