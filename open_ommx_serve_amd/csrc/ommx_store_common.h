// Argument block and arithmetic helpers shared by the store kernels (tuned 32x32 recipe kernel
// and the kernel for every other group size).  Every fp32 operation is a single IEEE rounding
// in the reference packer's order; the including files are compiled with -ffp-contract=off.
#pragma once
#include "ommx_common.h"
#include "ommx_rows.h"

namespace ommx {

struct StoreArgs {
    const void* K;
    const void* V;
    int64_t k_ts, k_hs, v_ts, v_hs;
    const int32_t* src_rows;
    const int32_t* dst_pages;
    const int32_t* dst_groups;
    const float* table;
    uint8_t* k_base;
    int8_t* k_scale;
    uint16_t* k_zp;
    uint16_t* k_ms;
    uint16_t* k_mc;
    uint8_t* k_obmp;        // index plane: bitmaps [G,H,D,4], or 7-bit streams [G,H,D,ceil(7k/8)]
    uint8_t* k_oval;
    uint8_t* v_main;
    int8_t* v_scale;
    uint16_t* v_zp;
    int32_t* err;
    int H, D, ps, kout;
    int v_vec;              // V rows allow 16-byte loads
    int idx_repr;           // 0 flat bitmap (codec.py:330-372), 1 relidx7 (pack.py:128-164)
    int select_abs;         // 0 signed top + bottom tails (pack.py:436-445), 1 largest |w| (pack.py:446-448)
    int scale_mode;         // 0 power of two, int8 exponent plane; 1 power of two, bf16 plane;
                            // 2 bf16((max - min) / 3) as it comes, bf16 plane (pack.py:459-463, 586-590)
    int gt, gc;             // tokens per K vector, channels per V vector (32 and 32 in the tuned kernel)
    int v_bf16;             // V is kept as bf16 rows [pages, ps, H, D]; v_scale = 1, v_zp = 0 (pack.py:596-602)
    int err_words;          // err is an array of OMMX_STORE_ERR_WORDS ints in host memory, one per bit, instead of one
                            // word of bits: the bus has no atomic OR, a store of 1 per bit needs none
    int32_t *own_pages, *own_groups;      // with a block of its own: its identity tables, written on the way instead of by a
                                          // launch of their own (4096-token block, whole call: 33.4 -> 31.9 us)
    int ring_span;          // rows of the ring the groups lie in (RingGroups)
    int groups;             // T / gt; workgroups beyond them copy rows into the history (bf16)
    BlockRows rows;
};

// Where a workgroup's place in the grid puts it.  Workgroups go to the eight dies (XCDs) in turn, each with an L2 of its own, and
// a token's row of a plane holds all heads side by side: 32 bytes of codes, 4 and 8 of steps and zero points a head.
// So the heads of eight groups are dispatched together, and the heads of one group to one die, whose L2 puts
// the lines together before they leave: x is 8 h + g % 8, y (and z, past 32768 of them) counts eights of groups.
// Groups side by side, as before, had the lines of a row written from eight dies one after the other, in pieces of 4 to
// 32 bytes: 32 K tokens of 8 heads into a pool 47.3 -> 43.0 us, with position streams 16 K 24.8 -> 23.4, at head_dim 64 32 K
// 31.8 -> 29.5, 64 x 64 vectors 32 K 52.7 -> 49.4.
// In line (x the group, y the head, z which of K and V): where the chip is half empty what counts is how soon the workgroups start,
// and these need nothing but their numbers for that.  Kernel alone, 8 heads, in line against by eights: 1 K tokens 5.6 / 5.8 us,
// 2 K 6.9 / 7.0, 4 K 7.3 / 7.6, but 6 K 11.4 / 11.1 and 8 K 13.6 / 13.3 (fp32 rows and other outlier counts: always); an instantiation of its own, as a test of which it is
// waits for the arguments (4 K 7.6).
// Rows of a prompt ride along with its packed groups: workgroups behind those of the groups copy a row each while the
// groups are still being packed.  A fresh prompt of 4096 rows, all of them kept: 7.3 + 9.1 us as two launches, 12.0 as one.
constexpr int kStoreEights = 32768;
enum StoreOrder { kByEights, kApartInLine, kApartByEights };      // apart: K and V in workgroups of their own
constexpr int kStoreInLine = 1024;                                 // groups and heads in line
struct StorePlace {
    int g, h;
    bool second;            // apart: the workgroup does V
};
// False when the workgroup has no group: it copied a row, or is beyond the last group.
template <StoreOrder ORDER>
__device__ __forceinline__ bool store_place(const StoreArgs& a, StorePlace& p) {
    constexpr bool APART = ORDER != kByEights;
    if constexpr (ORDER == kApartInLine) {
        const int past = static_cast<int>(blockIdx.z) - 2;
        if (past >= 0) {
            const int n = (past * a.H + static_cast<int>(blockIdx.y)) * a.groups + static_cast<int>(blockIdx.x);
            if (n < a.rows.rows) copy_block_row<false>(a.rows, n);
            return false;
        }
        p = {static_cast<int>(blockIdx.x), static_cast<int>(blockIdx.y), blockIdx.z == 1};
        return true;
    }
    const int eights = (a.groups + 7) >> 3, x = blockIdx.x;
    int e = static_cast<int>(blockIdx.z) * kStoreEights + static_cast<int>(blockIdx.y);
    const int past = e - (APART ? 2 : 1) * eights;
    if (past >= 0) {
        const int n = past * 8 * a.H + x;
        if (n < a.rows.rows) copy_block_row<false>(a.rows, n);
        return false;
    }
    p.second = APART && e >= eights;
    if (p.second) e -= eights;
    p.g = 8 * e + (x & 7);
    p.h = x >> 3;
    return p.g < a.groups;
}

// A workgroup each for K and V of a group and head?  Kernel alone, two against one, 8 heads: 5.9 against 6.5 us (1024 tokens), 6.8 / 8.1
// (2 K), 7.6 / 9.6 (4 K), 11.8 / 13.9 (6 K), 13.7 / 14.3 (8 K), 23.3 / 24.0 (16 K), 23.4 / 22.1 (16 K tokens into a pool); launches
// back to back fp32 rows 14.2 / 15.2 (1 K), 18.3 / 18.3 (4 K), 28.8 / 29.3 (8 K).  Past the line the chip is full either way, and the
// second workgroup is only one more to start.
constexpr int kStoreApart = 2048;
inline bool store_apart(const StoreArgs& a) { return a.groups * static_cast<int64_t>(a.H) <= kStoreApart; }
inline dim3 store_grid(const StoreArgs& a, StoreOrder order) {
    if (order == kApartInLine) {
        const int each = a.groups * a.H;
        return dim3(a.groups, a.H, 2 + (a.rows.rows + each - 1) / each);
    }
    const int64_t n = (order == kByEights ? 1 : 2) * ((a.groups + 7LL) / 8) + (a.rows.rows + 8LL * a.H - 1) / (8LL * a.H);
    return dim3(8 * a.H, static_cast<unsigned>(n < kStoreEights ? n : kStoreEights), static_cast<unsigned>((n + kStoreEights - 1) / kStoreEights));
}

// Entries of the identity tables that belong to K group g: the pages that begin in it, and its own.
__device__ __forceinline__ void write_own_tables(const StoreArgs& a, int g, int h, int tid) {
    if (!a.own_groups || h != 0) return;
    const int first = (g * a.gt + a.ps - 1) / a.ps, end = ((g + 1) * a.gt + a.ps - 1) / a.ps;
    for (int p = first + tid; p < end; p += blockDim.x) a.own_pages[p] = p;
    if (tid == 0) a.own_groups[g] = g;
}

// The bits a thread has found, into the caller's flag.  Reached on an error (or a noted wide step) only.
__device__ __forceinline__ void report_store_bits(const StoreArgs& a, int bits) {
    if (!a.err_words) { atomicOr(a.err, bits); return; }
    for (int i = 0; i < OMMX_STORE_ERR_WORDS; ++i)
        if ((bits >> i) & 1) *reinterpret_cast<volatile int32_t*>(a.err + i) = 1;
}


template <bool F32>
__device__ __forceinline__ float load_elem(const void* base, int64_t idx) {
    if (F32) return static_cast<const float*>(base)[idx];
    return bf16_to_f32(static_cast<const uint16_t*>(base)[idx]);
}

// rint(log2(x)) for x >= 1e-12 through the threshold table: the exponent of x's binade,
// plus one when x has reached that binade's rounding point.
__device__ __forceinline__ int pow2_round_exp(float x, const float* __restrict__ table) {
    const uint32_t kb = (__float_as_uint(x) >> 23) & 0xFFu;
    return static_cast<int>(kb) - 127 + (x >= table[kb] ? 1 : 0);
}

__device__ __forceinline__ float exp2_int(int e) {   // exact 2^e, e in [-126,127]
    return __uint_as_float(static_cast<uint32_t>(e + 127) << 23);
}

// The magnitude thresholds t[1..7] of the FP4 codes (ascending), the same for every thread, in scalar registers: left to the
// compiler they are read from memory again for every element of the general kernels, behind the copy of a row by vector loads.
// Launches back to back, 8 heads, with seven compares of values read again -> this, and the masks kept apart: 16 x 16
// vectors of four outliers 32 K tokens 111.6 -> 98.3 us, 64 x 32 of four 202 -> 166, 128 x 64 of eight 579 -> 538; small blocks of the
// tuned form as well, whose reads now start before the codes: 500 tokens into a pool, whole call, 17.4 -> 15.5.
__device__ __forceinline__ void fp4_boundaries(const float* __restrict__ tab, float (&t)[8]) {
    t[0] = 0.0f;
#pragma unroll
    for (int j = 1; j < 8; ++j) t[j] = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(tab[256 + j])));
}
// FP4 code of m: sign bit and the number of thresholds that |m| has reached, by three compares down the sorted ones.
__device__ __forceinline__ uint32_t fp4_encode(float m, const float (&t)[8]) {
    const float a = fabsf(m);
    const bool c4 = a >= t[4];
    const bool c2 = a >= (c4 ? t[6] : t[2]);
    const float lo = c4 ? t[5] : t[1], hi = c4 ? t[7] : t[3];
    const bool c1 = a >= (c2 ? hi : lo);
    return ((m < 0.0f) ? 8u : 0u) | (c4 ? 4u : 0u) | (c2 ? 2u : 0u) | (c1 ? 1u : 0u);
}

// x / 2^e is computed as x * 2^-e: 2^-e is exact for e in [-126,126], the product and the
// quotient are then the same real number, so they round alike, denormal results included.
// The quantisation step of one vector from raw = max(range, 1e-8) / 3 (pack.py:459-463).
struct Step {
    float scale;            // the step as the packer uses it (after its bf16 round trip)
    float inv;              // exact inverse when inv_ok
    bool inv_ok;
    int e;                  // exponent (power-of-two modes)
    uint16_t bits;          // the step as bf16
    bool in_range;
};
__device__ __forceinline__ Step make_step(float raw, int mode, const float* tab) {
    Step s;
    if (mode == 2) {
        s.bits = f32_to_bf16_rne(raw);
        s.scale = bf16_to_f32(s.bits);
        s.inv = 0.0f; s.inv_ok = false; s.e = 0; s.in_range = true;
        return s;
    }
    s.e = pow2_round_exp(fmaxf(raw, 1e-12f), tab);
    s.in_range = s.e >= -126 && s.e <= 127;
    s.scale = exp2_int(s.e);
    s.inv_ok = s.e >= -126 && s.e <= 126;
    s.inv = exp2_int(s.inv_ok ? -s.e : 0);
    s.bits = static_cast<uint16_t>((s.e + 127) << 7);
    return s;
}

// x / 3 rounded once, for x >= 1e-8 or infinite: a quotient within one unit and one exact remainder step, four instructions
// against the ten of a division by a variable (held against it for every mantissa).  The remainder of an infinity is NaN and
// is taken as a finite number, which leaves the infinity.
__device__ __forceinline__ float third(float x) {
    constexpr float r = 1.0f / 3.0f;
    const float q = x * r;
    return __builtin_fmaf(fmaxf(__builtin_fmaf(-3.0f, q, x), -3.0e38f), r, q);
}

// Ranks.  A bf16 value (in the high half of a word, the low half zero) as a two's complement number in the same place: zeros of
// both signs give 0, infinities and NaN lie at the ends.  Its inverse takes a key, whose low half holds a tie breaker.
__device__ __forceinline__ int rank_of(uint32_t b) {
    const int w = static_cast<int>(b), s = w >> 31;
    return (w ^ (s & 0x7FFFFFFF)) - s;
}
__device__ __forceinline__ float value_of_rank(int key) {
    const int v = key & static_cast<int>(0xFFFF0000u), s = v >> 31;
    return __int_as_float((v + s) ^ (s & 0x7FFFFFFF));
}
// The same for two values at once.
typedef int16_t s16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t ranks_of(uint32_t two) {
    const s16x2 s = __builtin_bit_cast(s16x2, two) >> s16x2{15, 15};
    const uint32_t x = (__builtin_bit_cast(uint32_t, s) & 0x7FFF7FFFu) ^ two;
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(s16x2, x) - s);
}
// Keys of the two: rank, and a tie breaker in the low half: a number below 64 that is known at compile time, or (_s) in a scalar
// register.  One instruction each, which the compiler would take apart to share the shift and the mask; `upper` is
// 0xFFFF0000 in a vector register (an instruction reads one scalar).
__device__ __forceinline__ int key_low(uint32_t two, int tie) {
    int k;
    asm("v_lshl_or_b32 %0, %1, 16, %2" : "=v"(k) : "v"(two), "n"(tie));
    return k;
}
__device__ __forceinline__ int key_high(uint32_t two, uint32_t upper, int tie) {
    int k;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(k) : "v"(two), "v"(upper), "n"(tie));
    return k;
}
__device__ __forceinline__ int key_low_s(uint32_t two, int tie) {
    int k;
    asm("v_lshl_or_b32 %0, %1, 16, %2" : "=v"(k) : "v"(two), "s"(tie));
    return k;
}
__device__ __forceinline__ int key_high_s(uint32_t two, uint32_t upper, int tie) {
    int k;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(k) : "v"(two), "v"(upper), "s"(tie));
    return k;
}
// Median, spelled out: where two of the three are known to be in order the compiler takes a minimum and a maximum instead.
__device__ __forceinline__ int med3_i32(int a, int b, int c) {
    int m;
    asm("v_med3_i32 %0, %1, %2, %3" : "=v"(m) : "v"(a), "v"(b), "v"(c));
    return m;
}
// N largest (smallest) keys in order from the end; the last one is the extreme of the rest.  `held` keys are there already
// (known at compile time while there are fewer than N).
template <int N>
__device__ __forceinline__ void keep_largest(int (&t)[N], int key, int held = N) {
    if (held > 0 && held < N) t[held] = min(t[held - 1], key);
#pragma unroll
    for (int j = N - 1; j > 0; --j)
        if (j < held) t[j] = med3_i32(t[j - 1], t[j], key);
    t[0] = held == 0 ? key : max(t[0], key);
}
template <int N>
__device__ __forceinline__ void keep_smallest(int (&t)[N], int key, int held = N) {
    if (held > 0 && held < N) t[held] = max(t[held - 1], key);
#pragma unroll
    for (int j = N - 1; j > 0; --j)
        if (j < held) t[j] = med3_i32(t[j - 1], t[j], key);
    t[0] = held == 0 ? key : min(t[0], key);
}

// INT2 code clamp(rint(x / 2^e), 0, 3) of a finite x.  v_cvt_pk_u8_f32 rounds to nearest even
// and saturates below at 0; the upper clamp commutes with the rounding.
__device__ __forceinline__ uint32_t int2_code(float x, float scale, float inv_scale, bool inv_ok) {
    if (inv_ok) return __builtin_amdgcn_cvt_pk_u8_f32(fminf(x * inv_scale, 3.0f), 0u, 0u);
    const float c = fminf(fmaxf(rintf(__fdiv_rn(x, scale)), 0.0f), 3.0f);
    return static_cast<uint32_t>(static_cast<int>(c));
}

// The same code from w, 2^-e and c = -zp * 2^-e in one fused multiply-add.  (w - zp) * 2^-e as the
// reference computes it is fl(w - zp) scaled exactly; the fused form rounds the exact (w - zp) * 2^-e
// once, and scaling by a power of two commutes with rounding while nothing under- or overflows: an
// underflowing quotient gives code 0 and an overflowing one code 3 either way.  The caller checks
// that c is finite (a huge zero point over a tiny step would make it infinite).
// (into byte `at` of `others`)
__device__ __forceinline__ uint32_t int2_code_fused(float w, float inv_scale, float c, uint32_t at = 0u, uint32_t others = 0u) {
    return __builtin_amdgcn_cvt_pk_u8_f32(fminf(__builtin_fmaf(w, inv_scale, c), 3.0f), at, others);
}

int launch_store_long(const StoreArgs& a, int T, int in_dtype, hipStream_t st);
int launch_store_generic(const StoreArgs& a, int T, int in_dtype, hipStream_t st);

}  // namespace ommx
