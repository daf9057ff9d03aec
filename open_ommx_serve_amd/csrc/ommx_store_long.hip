// Quantize-on-store for bf16 rows of the signed power-of-two recipes beside the serving one: K vectors
// of 32 / 64 / 128 tokens with 6 or 10 outliers (half of them from either end), V vectors of 32 / 64 / 128
// channels, dedicated or base-shared outlier map, either index plane, any head_dim that is a multiple of 32.
// Same planes and the same arithmetic as ommx_store_generic.hip (reference attention/pack.py:419-623), which
// keeps the recipes left over (other outlier counts, largest-magnitude selection, bf16 steps, fp32 rows, bf16 V).
//
// One workgroup of 2 D threads packs one (K group, kv head): the first D threads own one channel each and do K, the
// others take the V vectors meanwhile: 16 bytes a lane with the lanes of a load side by side, so that a vector lies in 4, 8
// or 16 neighbouring lanes, which exchange its extremes (DPP) and, one lane a vector, its step.  One thread a vector instead
// touched 64 cache lines a load and read each of them eight times, more than L1 holds: 32 K tokens of 64 x 64 vectors into a
// pool 76 -> 57 us, 1024 tokens 11.1 -> 9.9, 16 K tokens at head_dim 64 19.7 -> 17.8.  (The V rows are asked for when the K
// tile is there and are on their way during the selection; asked for before it they delay it, 57 -> 61 us.)
// The K tile comes in by 16-byte loads through LDS, and both passes over a
// channel (selection, codes) are loops that read it there: held in registers and unrolled, 128 tokens overrun the
// register file, and a straight-line body of 20-30 KB that every wave runs once is bound by instruction
// fetch.  Selection is what remains: the general kernel runs k passes of 5 instructions per element over
// the vector (64 tokens, 6 outliers: 1920); here one pass through two sorted networks of depth k/2 + 1
// (max / median of three on keys that hold the ordered bf16 value and the tie breaker) takes k + 7 an
// element and leaves the extremes of what stays as its last ranks.  The outliers come out of the network by
// rank and are wanted by position: each thread sorts them through its own few bytes of LDS.
#include <limits.h>

#include <utility>

#include "ommx_store_common.h"

namespace ommx {
namespace {

__device__ __forceinline__ int ordered_pair_half(uint32_t b) {      // b: a bf16 in the high half, low half zero
    const int s = static_cast<int>(b);
    return s ^ ((s >> 31) & 0x7FFF0000);
}
__device__ __forceinline__ float value_of_key(int k) {
    const int s = k & static_cast<int>(0xFFFF0000u);
    return __int_as_float(s ^ ((s >> 31) & 0x7FFF0000));
}
__device__ __forceinline__ int med3(int a, int b, int c) { return max(min(a, b), min(max(a, b), c)); }

// N largest keys in descending order; the last one is the largest of the rest
template <int N>
__device__ __forceinline__ void keep_largest(int (&t)[N], int key) {
#pragma unroll
    for (int j = N - 1; j > 0; --j) t[j] = med3(t[j - 1], t[j], key);
    t[0] = max(t[0], key);
}
template <int N>
__device__ __forceinline__ void keep_smallest(int (&t)[N], int key) {
#pragma unroll
    for (int j = N - 1; j > 0; --j) t[j] = med3(t[j - 1], t[j], key);
    t[0] = min(t[0], key);
}

// The extremes of bf16 values in packed 16-bit integers: b ^ (sign ? 0x7FFF : 0) orders them (-0 below +0, as v_min_f32 has
// it; infinities and NaN at the ends), two at once.
typedef int16_t s16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ s16x2 pair_image(uint32_t two) {
    const s16x2 m = __builtin_bit_cast(s16x2, two) >> s16x2{15, 15};
    return __builtin_bit_cast(s16x2, (__builtin_bit_cast(uint32_t, m) & 0x7FFF7FFFu) ^ two);
}
__device__ __forceinline__ float value_of_image(int img) {        // a sign-extended image
    return __int_as_float((img ^ ((img >> 31) & 0x7FFF)) << 16);
}
// (minimum, complement of the maximum) of a vector from those of its L neighbouring lanes, in all of them.
template <int CTRL>
__device__ __forceinline__ uint32_t with_lane(uint32_t x) {
    const uint32_t other = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(x), CTRL, 0xF, 0xF, true));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(s16x2, x), __builtin_bit_cast(s16x2, other)));
}
template <int L>
__device__ __forceinline__ uint32_t over_vector(uint32_t x) {
    x = with_lane<0xB1>(x);                          // quad_perm [1,0,3,2]
    x = with_lane<0x4E>(x);                          // quad_perm [2,3,0,1]
    if constexpr (L >= 8) x = with_lane<0x141>(x);   // row_half_mirror
    if constexpr (L >= 16) x = with_lane<0x140>(x);  // row_mirror
    return x;
}
// The value of lane N of the vector's L lanes.
template <int L, int N>
__device__ __forceinline__ float lane_of_vector(float x) {
    static_assert(L == 4 || L == 8 || L == 16, "lanes of a vector");
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, x), (N << 5) | (0x1F & ~(L - 1))));
}
template <int N, class F, int... I>
__device__ __forceinline__ void each_of(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, class F>
__device__ __forceinline__ void each(F&& f) { each_of<N>(f, std::make_integer_sequence<int, N>{}); }

// k_vec: K rows allow 16-byte loads.  As many waves a SIMD as the LDS allows (128 tokens: of head_dim 64), which the compiler
// has to be told: with the extremes of V in floats it took 78 to 256 registers by itself (64 tokens, 32 K into a pool 72 us
// instead of 61; 128 tokens at head_dim 64, 24 K into a block 40.6 instead of 36.7).  In packed integers they take a third of
// the registers and half of the instructions: 45 / 72 / 136, 11 K tokens at head_dim 64 14.4 -> 13.9 us.
template <int GT, int GC, int KH>
__global__ void __launch_bounds__(512, GT < GC ? 1 : GT == 32 ? 8 : GT == 64 ? 5 : 3) store_long_kernel(StoreArgs a, int k_vec) {
    constexpr int K = 2 * KH, MW = GT / 32, TIE = GT - 1;      // GT is a power of two: the tie breaker is its low bits
    constexpr int SORT = K <= 8 ? 8 : 12;                      // LDS bytes per thread and sorted list
    constexpr int NVAL = K / 2, NIDX = (7 * K + 7) / 8;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    StorePlace place;
    if (!store_place<kByEights>(a, place)) return;
    const int D = a.D, H = a.H, pieces = D >> 5;
    uint16_t* const s_k = reinterpret_cast<uint16_t*>(smem);   // [GT][D] the K tile
    uint8_t* const s_codes = smem + 2 * GT * D;                // [GT][D] one code per byte
    uint8_t* const s_pos = s_codes + GT * D;                   // [D][SORT] positions, then FP4 codes, by slot
    uint8_t* const s_fp4 = s_pos + SORT * D;
    uint8_t* const s_oval = s_fp4 + SORT * D;                  // [D][NVAL] as in memory
    uint8_t* const s_oidx = s_oval + 8 * D;                    // [D][bytes of the index plane] as in memory
    const int g = place.g, h = place.h, tid = threadIdx.x, NT = 2 * D;
    const int nidx = a.idx_repr == 0 ? GT / 8 : NIDX;
    const int64_t gs = a.dst_groups ? a.dst_groups[g] : g;
    const float* __restrict__ tab = a.table;
    int err = 0;
    auto src_row = [&](int i) -> int64_t { return a.src_rows ? a.src_rows[g * GT + i] : (int64_t)g * GT + i; };
    const int ps_log2 = __ffs(a.ps) - 1;                       // a divisor of GT: a power of two
    auto page_of = [&](int row) {
        const int lp = (g * GT + row) >> ps_log2;
        return a.dst_pages ? a.dst_pages[lp] : lp;
    };
    auto phys_row = [&](int page, int row) { return static_cast<int64_t>(page) * a.ps + (row & (a.ps - 1)); };

    // V: piece v_piece (8 channels) of rows v_row, v_row + 8, ... of the group
    constexpr int VP = GT / 8, VL = GC / 8;
    const int v = tid - D, v_row = v / (D / 8), v_piece = v % (D / 8);
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    typedef u32x4 u32x4_a2 __attribute__((aligned(2)));      // V rows need not be 16-byte aligned
    u32x4 vu[VP];
    const uint16_t* const v_base = static_cast<const uint16_t*>(a.V) + (int64_t)h * a.v_hs + 8 * v_piece;
    auto load_v = [&]() {
        int row[VP];
#pragma unroll
        for (int n = 0; n < VP; ++n) row[n] = g * GT + 8 * n + v_row;
        if (a.src_rows) {
#pragma unroll
            for (int n = 0; n < VP; ++n) row[n] = a.src_rows[row[n]];
        }
#pragma unroll
        for (int n = 0; n < VP; ++n) vu[n] = *reinterpret_cast<const u32x4_a2*>(v_base + row[n] * a.v_ts);
    };
    if (k_vec) {
        constexpr int KP = GT / 16;                // 16-byte pieces of the K tile a thread: rows k_row, k_row + 16, ...
        const int k_row = tid / (D / 8), c = 8 * (tid % (D / 8));
        const uint16_t* const base = static_cast<const uint16_t*>(a.K) + (int64_t)h * a.k_hs + c;
        uint4 ku[KP];
#pragma unroll
        for (int n = 0; n < KP; ++n) ku[n] = *reinterpret_cast<const uint4*>(base + src_row(16 * n + k_row) * a.k_ts);
#pragma unroll
        for (int n = 0; n < KP; ++n) *reinterpret_cast<uint4*>(s_k + (16 * n + k_row) * D + c) = ku[n];
    } else {
        for (int i = tid; i < GT * D; i += NT)
            s_k[i] = static_cast<const uint16_t*>(a.K)[src_row(i / D) * a.k_ts + (int64_t)h * a.k_hs + i % D];
    }
    __syncthreads();

    // ------------------------------------------------------------------ K vector
    if (tid < D) {
        const int d = tid;
        auto one = [&](int i) { return bf16_to_f32(s_k[i * D + d]); };       // token i of this thread's channel

        // (adding +0 turns -0 into +0: they tie in the reference's sorts)
        int t[KH + 1], b[KH + 1];
#pragma unroll
        for (int j = 0; j <= KH; ++j) { t[j] = INT_MIN; b[j] = INT_MAX; }
#pragma unroll 8
        for (int i = 0; i < GT; ++i) {
            const int ob = ordered_pair_half(__float_as_uint(one(i) + 0.0f));
            keep_largest(t, ob | (TIE - i));           // equal values: the lower position first
            keep_smallest(b, ob | i);
        }
#pragma unroll
        for (int j = 0; j <= KH; ++j) asm volatile("" : "+v"(t[j]), "+v"(b[j]));
        uint32_t top[MW], bot[MW], om[MW];
        auto mark = [&](uint32_t (&m)[MW], int pos) {
            const uint32_t bit = 1u << (pos & 31);
#pragma unroll
            for (int w = 0; w < MW; ++w) m[w] |= MW == 1 || (pos >> 5) == w ? bit : 0u;
        };
        bool clean = true;
#pragma unroll
        for (int w = 0; w < MW; ++w) top[w] = bot[w] = 0u;
#pragma unroll
        for (int j = 0; j < KH; ++j) { mark(top, TIE - (t[j] & TIE)); mark(bot, b[j] & TIE); }
#pragma unroll
        for (int w = 0; w < MW; ++w) clean = clean && (top[w] & bot[w]) == 0u;
        if (!clean) {
            // a top lane among the smallest (heavy ties): the reference takes the smallest of the vector with the
            // top lanes at +1e9 (pack.py:442-445)
            int c[KH];
#pragma unroll
            for (int j = 0; j < KH; ++j) c[j] = INT_MAX;
#pragma unroll
            for (int cc = 0; cc < MW; ++cc) {
#pragma unroll 1
                for (int i = 0; i < 32; ++i) {
                    const uint32_t bits = ((top[cc] >> i) & 1u) ? __float_as_uint(1e9f) & 0xFFFF0000u : __float_as_uint(one(32 * cc + i) + 0.0f);
                    keep_smallest(c, ordered_pair_half(bits) | i | (32 * cc));
                }
            }
#pragma unroll
            for (int w = 0; w < MW; ++w) bot[w] = 0u;
#pragma unroll
            for (int j = 0; j < KH; ++j) { b[j] = c[j]; mark(bot, c[j] & TIE); }
        }
        int picked = 0;
#pragma unroll
        for (int w = 0; w < MW; ++w) { om[w] = top[w] | bot[w]; picked += __popc(om[w]); }
        // NaN / Inf sort to the ends of the ordered keys
        if (!is_finite_f32(value_of_key(t[0])) || !is_finite_f32(value_of_key(b[0]))) err |= OMMX_ERR_NONFINITE_K;
        if (picked != K) err |= OMMX_ERR_UNDERFILLED;

        // affine base over the other lanes (pack.py:455-465): their extremes are the ranks after the chosen
        // ones.  A zero minimum, or zeros at both outlier ends, go the long way: which sign a zero result takes
        // depends on the lanes, not on the ranks.
        float mn = value_of_key(b[KH]), mx = value_of_key(t[KH]), omn = value_of_key(b[0]), omx = value_of_key(t[0]);
        if (!(clean && mn != 0.0f && (omn != 0.0f || omx != 0.0f))) {
            mn = 1e9f; mx = -1e9f; omn = 1e9f; omx = -1e9f;
#pragma unroll
            for (int c = 0; c < MW; ++c)
#pragma unroll 1
                for (int i = 0; i < 32; ++i) {
                    const bool o = (om[c] >> i) & 1u;
                    const float wi = one(32 * c + i);
                    mn = fminf(mn, o ? 1e9f : wi);
                    mx = fmaxf(mx, o ? -1e9f : wi);
                    omn = fminf(omn, o ? wi : 1e9f);
                    omx = fmaxf(omx, o ? wi : -1e9f);
                }
        }
        if (mn > 1e8f) mn = 0.0f;
        if (mx < -1e8f) mx = 0.0f;
        if (omn > 1e8f) omn = 0.0f;
        if (omx < -1e8f) omx = 0.0f;
        const Step st = make_step(__fdiv_rn(fmaxf(mx - mn, 1e-8f), 3.0f), 0, tab);
        if (!st.in_range) err |= OMMX_ERR_EXP_RANGE;
        if (st.e > 15) err |= OMMX_NOTE_WIDE_STEP;      // beyond the f16 operands of the matrix-core decode
        const uint16_t zp_b = f32_to_bf16_rne(mn);
        const float zp = bf16_to_f32(zp_b);

        const bool own_map = a.k_ms != nullptr;
        uint16_t mc_b = 0, ms_b = 0;
        float mc = 0.0f, ms = 0.0f;
        if (own_map) {       // pack.py:486-498; the step is a reciprocal and a product, two roundings (:492)
            mc_b = f32_to_bf16_rne(__fdiv_rn(omx + omn, 2.0f));
            ms_b = f32_to_bf16_rne(__fmul_rn(__fdiv_rn(1.0f, fmaxf(omx - omn, 1e-8f)), 12.0f));
            mc = bf16_to_f32(mc_b);
            ms = bf16_to_f32(ms_b);
        }
        const float zc = -zp * st.inv;
        const bool fused_k = st.inv_ok && fabsf(zc) < INFINITY;
        if (fused_k) {
#pragma unroll 8
            for (int i = 0; i < GT; ++i) s_codes[i * D + d] = static_cast<uint8_t>(int2_code_fused(one(i), st.inv, zc));
        } else {
#pragma unroll 1
            for (int i = 0; i < GT; ++i)
                s_codes[i * D + d] = static_cast<uint8_t>(int2_code(one(i) - zp, st.scale, st.inv, st.inv_ok));
        }

        // FP4 codes of the chosen lanes by slot = rank of their position.  |mapped| is largest at the extreme
        // lanes, which are chosen ones, so these decide whether every mapped value is finite (codec.py:55-57).
        float thr[8];
#pragma unroll
        for (int j = 1; j < 8; ++j)
            thr[j] = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(tab[256 + j])));
        thr[0] = 0.0f;
        bool mfin = true;
#pragma unroll
        for (int r = 0; r < K; ++r) {
            const int key = r < KH ? t[r] : b[r - KH];
            const int pos = r < KH ? TIE - (key & TIE) : key & TIE;
            const float wv = value_of_key(key);
            const float mapped = own_map ? (wv - mc) * ms : (st.inv_ok ? (wv - zp) * st.inv : __fdiv_rn(wv - zp, st.scale));
            mfin = mfin && is_finite_f32(mapped);
            int slot = 0;
#pragma unroll
            for (int w = 0; w < MW; ++w) {
                const uint32_t below = MW == 1 || (pos >> 5) == w ? (1u << (pos & 31)) - 1u : ((pos >> 5) > w ? 0xFFFFFFFFu : 0u);
                slot += __popc(om[w] & below);
            }
            slot = min(slot, SORT - 1);             // (an under-filled set is refused; its slots may repeat)
            s_pos[SORT * d + slot] = static_cast<uint8_t>(pos);
            s_fp4[SORT * d + slot] = static_cast<uint8_t>(fp4_encode_sorted(mapped, thr));
        }
        if (!mfin) err |= OMMX_ERR_NONFINITE_K;

        const int64_t gidx = (gs * H + h) * D + d;
        a.k_scale[gidx] = static_cast<int8_t>(st.e);
        a.k_zp[gidx] = zp_b;
        if (own_map) { a.k_ms[gidx] = ms_b; a.k_mc[gidx] = mc_b; }

        // this thread's own bytes back in slot order (one wave writes and reads them: program order is enough)
        uint32_t pw[SORT / 4], fw[SORT / 4];
#pragma unroll
        for (int w = 0; w < SORT / 4; ++w) {
            pw[w] = *reinterpret_cast<const uint32_t*>(s_pos + SORT * d + 4 * w);
            fw[w] = *reinterpret_cast<const uint32_t*>(s_fp4 + SORT * d + 4 * w);
        }
        uint64_t nib = 0, lo = 0, hi = 0;           // position s at bits [7s, 7s+7) of hi:lo
#pragma unroll
        for (int s = 0; s < K; ++s) {
            const uint64_t pos = (pw[s >> 2] >> (8 * (s & 3))) & 0x7Fu;
            nib |= static_cast<uint64_t>((fw[s >> 2] >> (8 * (s & 3))) & 0xFu) << (4 * s);
            if (7 * s < 64) lo |= pos << (7 * s);
            if (7 * s + 7 > 64) hi |= 7 * s >= 64 ? pos << (7 * s - 64) : pos >> (64 - 7 * s);
        }
#pragma unroll
        for (int q = 0; q < NVAL; ++q) s_oval[d * NVAL + q] = static_cast<uint8_t>(nib >> (8 * q));
        if (a.idx_repr == 0) {
#pragma unroll
            for (int w = 0; w < MW; ++w) reinterpret_cast<uint32_t*>(s_oidx)[d * MW + w] = om[w];
        } else {
#pragma unroll
            for (int q = 0; q < NIDX; ++q)
                s_oidx[d * NIDX + q] = static_cast<uint8_t>(q < 8 ? lo >> (8 * q) : hi >> (8 * (q - 8)));
        }
    } else {
        // -------------------------------------------- V vectors (pack.py:604-623)
        load_v();
        // (minimum, complement of the maximum) of a piece, then of its vector in all VL lanes
        uint32_t ends[VP];
#pragma unroll
        for (int n = 0; n < VP; ++n) {
            const u32x4 w = vu[n];
            s16x2 lo = pair_image(w[0]), hi = lo;
#pragma unroll
            for (int c = 1; c < 4; ++c) {
                const s16x2 img = pair_image(w[c]);
                lo = __builtin_elementwise_min(lo, img);
                hi = __builtin_elementwise_max(hi, img);
            }
            const uint32_t l = __builtin_bit_cast(uint32_t, lo), h2 = ~__builtin_bit_cast(uint32_t, hi);
            const s16x2 even = __builtin_bit_cast(s16x2, __builtin_amdgcn_perm(h2, l, 0x05040100u)),
                        odd = __builtin_bit_cast(s16x2, __builtin_amdgcn_perm(h2, l, 0x07060302u));
            ends[n] = over_vector<VL>(__builtin_bit_cast(uint32_t, __builtin_elementwise_min(even, odd)));
        }
        // Lane i of a vector's VL lanes works out the step of the vector of turn VL r + i, for all of them.
        const int me = v % VL, ngv = D / GC;
        int page[VP];
#pragma unroll
        for (int n = 0; n < VP; ++n) page[n] = page_of(8 * n + v_row);
        auto code_word = [&](int pg, int row) -> uint16_t& {
            return reinterpret_cast<uint16_t*>(a.v_main + (phys_row(pg, row) * H + h) * (D / 4))[v_piece];
        };
#pragma unroll
        for (int r = 0; r < VP; r += VL) {
            uint32_t mine = ends[r];
#pragma unroll
            for (int n = 1; n < VL && r + n < VP; ++n) mine = me == n ? ends[r + n] : mine;
            const float my_mn = value_of_image(static_cast<int16_t>(mine)), my_mx = value_of_image(static_cast<int16_t>(~mine >> 16));
            if (!is_finite_f32(my_mn) || !is_finite_f32(my_mx)) err |= OMMX_ERR_NONFINITE_V;
            const Step st = make_step(__fdiv_rn(fmaxf(my_mx - my_mn, 1e-8f), 3.0f), 0, tab);
            const uint16_t zp_b = f32_to_bf16_rne(my_mn);
            const float zc = -bf16_to_f32(zp_b) * st.inv;
            if (r + me < VP) {
                if (!st.in_range) err |= OMMX_ERR_EXP_RANGE;
                if (st.e > 15) err |= OMMX_NOTE_WIDE_STEP;
                const int64_t vidx = (phys_row(page_of(8 * (r + me) + v_row), 8 * (r + me) + v_row) * H + h) * ngv + v_piece / VL;
                a.v_scale[vidx] = static_cast<int8_t>(st.e);
                a.v_zp[vidx] = zp_b;
            }
            const float my_inv = st.inv_ok && fabsf(zc) < INFINITY ? st.inv : 0.0f;       // 0: the long way, below
            each<(VP < VL ? VP : VL)>([&](auto turn) {
                constexpr int n = decltype(turn)::value;
                const int at = r + n;
                const float inv = lane_of_vector<VL, n>(my_inv), c0 = lane_of_vector<VL, n>(zc);
                const u32x4 w = vu[at];
                uint32_t bits = 0;
#pragma unroll
                for (int f = 0; f < 2; ++f) {
                    uint32_t four = 0;
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const uint32_t x = w[2 * f + (c >> 1)];
                        const float val = __uint_as_float((c & 1) ? x & 0xFFFF0000u : x << 16);
                        four = __builtin_amdgcn_cvt_pk_u8_f32(fminf(__builtin_fmaf(val, inv, c0), 3.0f), c, four);
                    }
                    bits |= __builtin_amdgcn_udot4(four, 0x40100401u, 0u, false) << (8 * f);
                }
                if (inv != 0.0f) code_word(page[at], 8 * at + v_row) = static_cast<uint16_t>(bits);
                asm volatile("" : : : "memory");       // addresses of the next turn: in the next turn
            });
            if (__ballot(my_inv == 0.0f) != 0) {       // steps or zero points at the ends of the range: read again, one by one
#pragma unroll 1
                for (int n = 0; n < VL && r + n < VP; ++n) {
                    const int from = (static_cast<int>(threadIdx.x) & 63 & ~(VL - 1)) + n, row = 8 * (r + n) + v_row;
                    const float lo = __shfl(my_mn, from), hi = __shfl(my_mx, from), inv = __shfl(my_inv, from);
                    if (inv != 0.0f) continue;
                    const Step s1 = make_step(__fdiv_rn(fmaxf(hi - lo, 1e-8f), 3.0f), 0, tab);
                    const float zp = bf16_to_f32(f32_to_bf16_rne(lo));
                    const uint16_t* const e = v_base + src_row(row) * a.v_ts;
                    uint32_t bits = 0;
#pragma unroll 1
                    for (int c = 0; c < 8; ++c)
                        bits |= int2_code(bf16_to_f32(e[c]) - zp, s1.scale, s1.inv, s1.inv_ok) << (2 * c);
                    code_word(page_of(row), row) = static_cast<uint16_t>(bits);
                }
            }
        }
    }
    __syncthreads();

    {   // D frames of NVAL / nidx bytes each, contiguous in memory: whole dwords
        const int64_t obase = (gs * H + h) * (int64_t)D * NVAL;
        for (int wd = tid; wd < D * NVAL / 4; wd += NT)
            reinterpret_cast<uint32_t*>(a.k_oval + obase)[wd] = reinterpret_cast<const uint32_t*>(s_oval)[wd];
        const int64_t ibase = (gs * H + h) * (int64_t)D * nidx;
        for (int wd = tid; wd < D * nidx / 4; wd += NT)
            reinterpret_cast<uint32_t*>(a.k_obmp + ibase)[wd] = reinterpret_cast<const uint32_t*>(s_oidx)[wd];
    }

    // ------------------------------------------------- k_base rows: 8 bytes = 32 channels a piece
    for (int it = tid; it < GT * pieces; it += NT) {
        const int tk = it / pieces, j = it % pieces;
        uint64_t kb8 = 0;
        const uint4* cr = reinterpret_cast<const uint4*>(s_codes + tk * D + 32 * j);
#pragma unroll
        for (int q4 = 0; q4 < 2; ++q4) {
            const uint4 u = cr[q4];
            const uint32_t uw[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
            for (int q = 0; q < 4; ++q)
                kb8 |= static_cast<uint64_t>(__builtin_amdgcn_udot4(uw[q], 0x40100401u, 0u, false)) << (8 * (4 * q4 + q));
        }
        reinterpret_cast<uint64_t*>(a.k_base)[(phys_row(page_of(tk), tk) * H + h) * pieces + j] = kb8;
    }

    write_own_tables(a, g, h, tid);
    if (err && a.err) report_store_bits(a, err);
}

template <int GT, int GC>
int launch_k(const StoreArgs& a, int T, hipStream_t st) {
    const dim3 grid = store_grid(a, kByEights), block(2 * a.D);
    const size_t shm = static_cast<size_t>(a.D) * (3 * GT + 2 * 12 + 8 + 16);
    if (shm > 64 * 1024) return 1;           // 128 tokens of a 256-channel head: the general kernel
    const int k_vec = reinterpret_cast<uintptr_t>(a.K) % 16 == 0 && a.k_ts % 8 == 0 && a.k_hs % 8 == 0;
    if (a.kout == 6) hipLaunchKernelGGL((store_long_kernel<GT, GC, 3>), grid, block, shm, st, a, k_vec);
    else hipLaunchKernelGGL((store_long_kernel<GT, GC, 5>), grid, block, shm, st, a, k_vec);
    return 0;
}
template <int GT>
int launch_gc(const StoreArgs& a, int T, hipStream_t st) {
    switch (a.gc) {
        case 32: return launch_k<GT, 32>(a, T, st);
        case 64: return launch_k<GT, 64>(a, T, st);
        case 128: return launch_k<GT, 128>(a, T, st);
    }
    return 1;
}

}  // namespace

// 0 launched, 1 when the recipe belongs to another kernel.  6 and 10 outliers are what the named recipes use; a wider
// choice would add an instantiation per count for recipes nobody serves.
int launch_store_long(const StoreArgs& a, int T, int in_dtype, hipStream_t st) {
    if (in_dtype != 0 || a.select_abs || a.scale_mode != 0 || a.v_bf16 || (a.kout != 6 && a.kout != 10) || a.D % 32 ||
        a.D > 256 || a.gt % a.ps)
        return 1;
    switch (a.gt) {
        case 32: return launch_gc<32>(a, T, st);
        case 64: return launch_gc<64>(a, T, st);
        case 128: return launch_gc<128>(a, T, st);
    }
    return 1;
}

}  // namespace ommx
