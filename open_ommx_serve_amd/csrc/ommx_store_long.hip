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
// The K tile comes in by 16-byte loads through LDS, two tokens of a channel a word, and both passes over a
// channel (selection, codes) are loops that read it there: held in registers and unrolled, 128 tokens overrun the
// register file, and a straight-line body of 20-30 KB that every wave runs once is bound by instruction
// fetch.  Selection is what remains: the general kernel runs k passes of 5 instructions per element over
// the vector (64 tokens, 6 outliers: 1920); here one pass through two sorted networks of depth k/2 + 1
// (max / median of three on keys that hold the rank of the bf16 value and the tie breaker; ranks of two tokens at
// once) takes k + 5 an element and leaves the extremes of what stays as its last ranks.  The outliers come out of the
// network by rank and are wanted by position: position and FP4 code go through a fixed sorting network as one number.
// The codes of two tokens take the place of the tokens in the tile.  (32 K tokens into a pool, a token a halfword,
// codes in a tile of their own and the outliers sorted through LDS -> this: 64 x 64 vectors with six outliers 49.4 ->
// 45.7 us, 128 x 128 with ten 78.6 -> 54.1, which also has four workgroups a compute unit instead of two; 8 K tokens
// 17.4 -> 16.2 and 24.3 -> 21.4; 11 K at head_dim 64 16.5 -> 15.1.)
#include <limits.h>

#include <utility>

#include "ommx_store_common.h"

namespace ommx {
namespace {

// Ascending order by a fixed network of compare-exchanges: the smallest known ones, 12 for six and 29 for ten (Knuth, The Art of
// Computer Programming, vol. 3, 5.3.4), in the layers that Bert Dobbelaere's list of sorting networks gives.
__device__ __forceinline__ void in_order(int& a, int& b) {
    const int lo = min(a, b);
    b = max(a, b);
    a = lo;
}
__device__ __forceinline__ void sort_ascending(int (&x)[6]) {
    constexpr int net[12][2] = {{0, 5}, {1, 3}, {2, 4}, {1, 2}, {3, 4}, {0, 3}, {2, 5}, {0, 1}, {2, 3}, {4, 5}, {1, 2}, {3, 4}};
#pragma unroll
    for (int i = 0; i < 12; ++i) in_order(x[net[i][0]], x[net[i][1]]);
}
__device__ __forceinline__ void sort_ascending(int (&x)[10]) {
    constexpr int net[29][2] = {{0, 8}, {1, 9}, {2, 7}, {3, 5}, {4, 6}, {0, 2}, {1, 4}, {5, 8}, {7, 9}, {0, 3},
                                {2, 4}, {5, 7}, {6, 9}, {0, 1}, {3, 6}, {8, 9}, {1, 5}, {2, 3}, {4, 8}, {6, 7},
                                {1, 2}, {3, 5}, {4, 6}, {7, 8}, {2, 3}, {4, 5}, {6, 7}, {3, 4}, {5, 6}};
#pragma unroll
    for (int i = 0; i < 29; ++i) in_order(x[net[i][0]], x[net[i][1]]);
}

// The extremes of bf16 values in packed 16-bit integers: b ^ (sign ? 0x7FFF : 0) orders them (-0 below +0, as v_min_f32 has
// it; infinities and NaN at the ends), two at once.
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

// k_vec: K rows allow 16-byte loads.  As many waves a SIMD as the LDS allows (128 tokens: four, with up to nine registers in
// scratch memory; with three and none 32 K tokens into a pool take 56.5 us instead of 54.1), which the compiler has to be
// told: with the extremes of V in floats it took 78 to 256 registers by itself.  In packed integers they take a third of
// the registers and half of the instructions.
template <int GT, int GC, int KH>
__global__ void __launch_bounds__(512, GT < GC ? 1 : GT == 32 ? 8 : GT == 64 ? 7 : 4) store_long_kernel(StoreArgs a, int k_vec) {
    constexpr int K = 2 * KH, MW = GT / 32, TIE = GT - 1;      // GT is a power of two: the tie breaker is its low bits
    constexpr int NVAL = K / 2, NIDX = (7 * K + 7) / 8;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    StorePlace place;
    if (!store_place<kByEights>(a, place)) return;
    const int D = a.D, H = a.H, pieces = D >> 5;
    uint32_t* const s_k = reinterpret_cast<uint32_t*>(smem);   // [GT / 2][D] the K tile, two tokens of a channel a word; then their
                                                               // two codes in the word's lower bytes
    uint8_t* const s_oval = smem + 2 * GT * D;                 // [D][NVAL] as in memory
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
        constexpr int KP = GT / 32;                // 16-byte pieces of two rows a thread: pairs k_row, k_row + 16, ...
        const int k_row = tid / (D / 8), c = 8 * (tid % (D / 8));
        const uint16_t* const base = static_cast<const uint16_t*>(a.K) + (int64_t)h * a.k_hs + c;
        u32x4 ku[KP][2];
#pragma unroll
        for (int n = 0; n < KP; ++n)
#pragma unroll
            for (int o = 0; o < 2; ++o) ku[n][o] = *reinterpret_cast<const u32x4*>(base + src_row(2 * (16 * n + k_row) + o) * a.k_ts);
#pragma unroll
        for (int n = 0; n < KP; ++n) {
            u32x4* const to = reinterpret_cast<u32x4*>(s_k + (16 * n + k_row) * D + c);
#pragma unroll
            for (int q = 0; q < 2; ++q) {          // channels c + 4q .. c + 4q + 3
                u32x4 w;
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    w[2 * e] = __builtin_amdgcn_perm(ku[n][1][2 * q + e], ku[n][0][2 * q + e], 0x05040100u);
                    w[2 * e + 1] = __builtin_amdgcn_perm(ku[n][1][2 * q + e], ku[n][0][2 * q + e], 0x07060302u);
                }
                to[q] = w;
            }
        }
    } else {
        for (int i = tid; i < GT * D; i += NT)
            reinterpret_cast<uint16_t*>(s_k)[2 * ((i / D >> 1) * D + i % D) + (i / D & 1)] =
                static_cast<const uint16_t*>(a.K)[src_row(i / D) * a.k_ts + (int64_t)h * a.k_hs + i % D];
    }
    __syncthreads();

    // ------------------------------------------------------------------ K vector
    if (tid < D) {
        const int d = tid;
        auto two = [&](int i) { return s_k[i * D + d]; };                    // tokens 2i and 2i + 1 of this thread's channel
        auto one = [&](int i) { return bf16_to_f32(reinterpret_cast<const uint16_t*>(s_k)[2 * ((i >> 1) * D + d) + (i & 1)]); };

        int t[KH + 1], b[KH + 1];
        uint32_t upper = 0xFFFF0000u;
        asm("" : "+v"(upper));
#pragma unroll
        for (int j = 0; j <= KH; ++j) { t[j] = INT_MIN; b[j] = INT_MAX; }
#pragma unroll 4
        for (int i = 0; i < GT; i += 2) {
            const uint32_t y = ranks_of(two(i >> 1));  // (zeros of both signs have one rank: they tie in the reference's sorts)
            keep_largest(t, key_low_s(y, TIE - i));      // equal values: the lower position first
            keep_smallest(b, key_low_s(y, i));
            keep_largest(t, key_high_s(y, upper, TIE - i - 1));
            keep_smallest(b, key_high_s(y, upper, i + 1));
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
                    const uint32_t bits = ((top[cc] >> i) & 1u) ? __float_as_uint(1e9f) & 0xFFFF0000u : __float_as_uint(one(32 * cc + i));
                    keep_smallest(c, rank_of(bits) | i | (32 * cc));
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
        if (!is_finite_f32(value_of_rank(t[0])) || !is_finite_f32(value_of_rank(b[0]))) err |= OMMX_ERR_NONFINITE_K;
        if (picked != K) err |= OMMX_ERR_UNDERFILLED;

        // affine base over the other lanes (pack.py:455-465): their extremes are the ranks after the chosen
        // ones.  A zero minimum, or zeros at both outlier ends, go the long way: which sign a zero result takes
        // depends on the lanes, not on the ranks.
        float mn = value_of_rank(b[KH]), mx = value_of_rank(t[KH]), omn = value_of_rank(b[0]), omx = value_of_rank(t[0]);
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
        const Step st = make_step(third(fmaxf(mx - mn, 1e-8f)), 0, tab);
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
#pragma unroll 4
            for (int i = 0; i < GT / 2; ++i) {
                const uint32_t w = two(i);
                const uint32_t even = int2_code_fused(__uint_as_float(w << 16), st.inv, zc);
                s_k[i * D + d] = int2_code_fused(__uint_as_float(w & 0xFFFF0000u), st.inv, zc, 1, even);
            }
        } else {
#pragma unroll 1
            for (int i = 0; i < GT / 2; ++i)
                s_k[i * D + d] = int2_code(one(2 * i) - zp, st.scale, st.inv, st.inv_ok) |
                                 int2_code(one(2 * i + 1) - zp, st.scale, st.inv, st.inv_ok) << 8;
        }

        // FP4 codes of the chosen lanes, in the order of their positions: position and code as one number, sorted.  |mapped| is
        // largest at the extreme lanes, which are chosen ones, so these decide whether every mapped value is finite
        // (codec.py:55-57).
        float thr[8];
        fp4_boundaries(tab, thr);
        bool mfin = true;
        int slot[K];
#pragma unroll
        for (int r = 0; r < K; ++r) {
            const int key = r < KH ? t[r] : b[r - KH];
            const int pos = r < KH ? TIE - (key & TIE) : key & TIE;
            const float wv = value_of_rank(key);
            const float mapped = own_map ? (wv - mc) * ms : (st.inv_ok ? (wv - zp) * st.inv : __fdiv_rn(wv - zp, st.scale));
            if (r % KH == 0) mfin = mfin && is_finite_f32(mapped);
            slot[r] = pos << 5 | (r < KH ? 0 : 16) | static_cast<int>(fp4_encode(mapped, thr));
        }
        sort_ascending(slot);
        if (picked != K) {          // positions taken from both ends (reported): each once, with its code from the lower end; then the last again
#pragma unroll
            for (int s = 0; s + 1 < K; ++s)
                if (slot[s] >> 5 == slot[s + 1] >> 5) slot[s] = INT_MAX;
            sort_ascending(slot);
#pragma unroll
            for (int s = 1; s < K; ++s)
                if (slot[s] == INT_MAX) slot[s] = slot[s - 1];
        }
        if (!mfin) err |= OMMX_ERR_NONFINITE_K;

        const int64_t gidx = (gs * H + h) * D + d;
        a.k_scale[gidx] = static_cast<int8_t>(st.e);
        a.k_zp[gidx] = zp_b;
        if (own_map) { a.k_ms[gidx] = ms_b; a.k_mc[gidx] = mc_b; }

        uint64_t nib = 0, lo = 0, hi = 0;           // position s at bits [7s, 7s+7) of hi:lo
#pragma unroll
        for (int s = 0; s < K; ++s) {
            const uint64_t pos = static_cast<uint32_t>(slot[s]) >> 5;
            nib |= static_cast<uint64_t>(slot[s] & 0xF) << (4 * s);
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
            const Step st = make_step(third(fmaxf(my_mx - my_mn, 1e-8f)), 0, tab);
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
                    const Step s1 = make_step(third(fmaxf(hi - lo, 1e-8f)), 0, tab);
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

    // ------------------------------------------------- k_base rows: 4 bytes = 16 channels a piece, of two tokens
    for (int it = tid; it < GT / 2 * 2 * pieces; it += NT) {
        const int tp = it / (2 * pieces), j = it % (2 * pieces), turn = (j >> 1) & 3;
        // 16 words, four at a time; the pieces start in turn, so that neighbouring lanes read from different banks
        const u32x4* const words = reinterpret_cast<const u32x4*>(s_k + tp * D + 16 * j);
        uint32_t four[4];                          // bytes 0 and 1: four codes of either token
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const u32x4 w = words[(q + turn) & 3];
            four[q] = w[0] | w[1] << 2 | w[2] << 4 | w[3] << 6;
        }
        const uint32_t lo = __builtin_amdgcn_perm(four[1], four[0], 0x05010400u), hi = __builtin_amdgcn_perm(four[3], four[2], 0x05010400u);
        const uint32_t even = __builtin_amdgcn_perm(hi, lo, 0x05040100u), odd = __builtin_amdgcn_perm(hi, lo, 0x07060302u);
        const int back = (32 - 8 * turn) & 31;     // byte q is piece (q + turn) % 4
        const int page = page_of(2 * tp);          // (a page holds an even number of tokens, or one)
        reinterpret_cast<uint32_t*>(a.k_base)[(phys_row(page, 2 * tp) * H + h) * 2 * pieces + j] = __builtin_amdgcn_alignbit(even, even, back);
        reinterpret_cast<uint32_t*>(a.k_base)[(phys_row(a.ps == 1 ? page_of(2 * tp + 1) : page, 2 * tp + 1) * H + h) * 2 * pieces + j] =
            __builtin_amdgcn_alignbit(odd, odd, back);
    }

    write_own_tables(a, g, h, tid);
    if (err && a.err) report_store_bits(a, err);
}

template <int GT, int GC>
int launch_k(const StoreArgs& a, int T, hipStream_t st) {
    const dim3 grid = store_grid(a, kByEights), block(2 * a.D);
    const size_t shm = static_cast<size_t>(a.D) * (2 * GT + 8 + 16);
    if (GT == 128 && a.D > 128) return 1;    // (LDS: the general kernel)
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
