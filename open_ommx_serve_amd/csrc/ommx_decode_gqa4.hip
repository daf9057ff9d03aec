// Split-KV decode kernel for gfx950, serving shape: head_dim 128, 1, 2, 4 or 8 q heads per kv head,
// 6 outliers per K vector of 32 tokens (either index plane, either outlier map), INT2 V with
// 32-channel vectors, int8 exponents; in a general form (GEN) also 1..8 outliers on the bitmap
// plane and head_dim 64 with 1, 2 or 4 q heads per kv head; and (GTS) K vectors of 64 or 128 tokens on
// the position-stream plane with 4 or 8 q heads per kv head, 6 outliers or 10 of 128.  Same operator as
// ommx_gpu_serve/attention/paged_decode.py:1255-2284; the other shapes of the matrix-core path
// (no outliers, planes of 4 GiB and more or of unknown extent) stay on the kernel in ommx_decode.hip.
//
// A wavefront owns one kv head (and its q heads) of one split and walks it 64 tokens at a time;
// a workgroup is 4 waves = 4 neighbouring kv heads.  Measured on MI355X this operator is bound
// by how many instructions a SIMD can issue (vector ALU first, LDS second, a 16-byte LDS access
// taking four issue slots), so the kernel is built for few instructions per token and to keep
// THREE waves per SIMD resident (two with longer groups or eight outlier slots): at most 168 vector registers, no scratch memory,
// 13.4 KB of LDS per wave.  What that takes, against the kernel in ommx_decode.hip:
//   * P.V runs transposed (rows = V channels, columns = q heads), the V step 2^e sits in the
//     exponent field of the V operand, and the four column replicas of the q heads each take
//     every fourth channel block, so the output accumulator is 8 registers instead of 32;
//   * the softmax denominator comes out of the same matrix instruction that sums p*2^e and
//     p*zp (a row of ones), the running maximum is refreshed only when a logit exceeds it by
//     more than 2^8 (any bound that keeps exp2 in range serves an online softmax);
//   * the V staging area of LDS is the K staging area of the same step, reused once QK is done.
// With 8 q heads per kv head (NH = 8) the sixteen matrix rows / columns are two replicas of the
// heads instead of four: a lane then keeps four heads of one token of either group, the output
// takes four accumulators, and two workgroups fit a compute unit (184 to 197 registers, 14.1 KB of LDS
// per wave); everything up to the logits is the same code.
// Arithmetic: exact 16-bit operands, fp32 accumulation, as in ommx_decode.hip.
//   A (QK)   q * 2^(10-2m) as f16 in pair order, m = 2..4 (3 or 4 with longer groups) fixed per channel pair; this one operand
//            set serves the base codes, the outlier tile and the bias columns.
//   K base   B = (1 + code*2^(2m-10)) * 2^e as f16: the 2-bit code is dropped into mantissa bits
//            [2m+1:2m] of a per-(group, channel) pattern that carries the exponent, one and-or per
//            channel pair.  The constant terms sum q*zp and sum A*2^e come from one small "bias"
//            MFMA per 64 tokens (zero points are staged divided by the channel's 2^(10-2m), exact).
//   outliers a channel-major pass (one lane = two channels) reads the stored 2-bit code of every
//            outlier position back from the staged K rows (the base MFMA takes every position as
//            stored; nothing is cleared there) and scatters
//            (outlier - zp - code*2^e) / 2^(10-2m) as f16 into a [32 tokens][128 channels] tile
//            that is the B operand of an f16 MFMA against the same A.  Entries whose f16 rounding
//            could show on a logit add their rounding residual times q through LDS float atomics.
//   P.V      A = (1 + code/4 | 1 + code/16) * 2^e_v as f16 for 8 tokens of one channel (longer groups code/4), B = p (f16).
#include <type_traits>

#include "ommx_decode_recipe.h"
#include "ommx_decode_shares.h"
#include "ommx_decode_tail.h"
#include "ommx_decode_util.h"

namespace ommx {

namespace {

using namespace decode_util;

// The kernels that also attend the tail rows are compiled apart (ommx_decode_gqa4_tail.hip): the tail's code beside the
// splits' costs a launch that does not need it 0.3 to 1 % (registers, spilled scalars).
#ifndef OMMX_GQA4_LAUNCH
#define OMMX_GQA4_LAUNCH launch_decode_gqa4
constexpr bool TAIL = false;
#else
constexpr bool TAIL = true;
#endif

#ifndef OMMX_GQA4_WAVES
#define OMMX_GQA4_WAVES 3          // waves per SIMD the register budget is set for
#endif
constexpr int D = 128;
// ---- per-wave LDS map (bytes) ------------------------------------------------------------
constexpr int TILE_ROW = 272;                       // bytes per row of the outlier tile (256 used)
constexpr int KT_ROW = 40;                          // bytes per staged K code row (32 used): 16 rows read as b64 spread over all banks
constexpr int VT_COL = 68;                          // dwords per V dword column (64 used)
constexpr int PT_ROW = 72;                          // halfwords per row of the f16 [row][64 tokens] arrays
// Regions, in an order that makes row -1 of the tile, of the corrections and of the K codes harmless: the lowest bit of an empty
// bitmap is -1 (lowest_bit), and a map with fewer bits than outlier slots is something a caller's planes can hold (the store
// writes one, and reports it, for a K vector without enough distinct values; a converted index plane has zeros for a bad
// vector).  A code row -1 is read from the wave's own constant rows, a tile row -1 is written over staged V that nobody reads
// any more, corrections of a row -1 go to the unused end of the tile's last row: the neighbouring wave, another kv head, is not
// touched, and no position needs an instruction for it (a test where corrections are added, which most groups do for some
// entry, cost 1 % at 64 K).
// They depend on the number of q heads per kv head (NH = 4 or 8) and, with groups longer than 32 tokens, on one
// more row of the tile: where the outliers of the group's other tokens go.
template <int NH, bool LONG>
struct LdsMap {
    static constexpr int OFF_ZERO = 0;                         // 128 B of zeros, never written again
    static constexpr int OFF_ONES = OFF_ZERO + 128;            // 128 B of f16 1.0, never written again
    static constexpr int OFF_KT = OFF_ONES + 128;              // [64 tokens][KT_ROW] K code rows
    static constexpr int OFF_MAG = OFF_KT + 64 * KT_ROW;       // [2 groups][128] f16 2^e, channels (p, p+8) adjacent
    static constexpr int OFF_ZPP = OFF_MAG + 512;              // same order, f16 zero points over the A scale
    // after QK the same bytes hold what P.V needs
    static constexpr int OFF_VT = OFF_KT;                      // [8 dword columns][VT_COL] V code dwords
    static constexpr int OFF_PT = OFF_VT + 8 * VT_COL * 4;     // [NH heads][PT_ROW] f16 softmax weights
    static constexpr int OFF_VZ = OFF_PT + NH * PT_ROW * 2;    // [4 channel groups][PT_ROW] f16 V zero points
    static constexpr int OFF_VS = OFF_VZ + 4 * PT_ROW * 2;     // [4 channel groups][PT_ROW] f16 2^e_v
    static constexpr int OFF_TILE = OFF_VS + 4 * PT_ROW * 2;   // [32 tokens][TILE_ROW] f16 outlier deltas of one group
    static constexpr int TILE_END = OFF_TILE + (LONG ? 33 : 32) * TILE_ROW;
    static constexpr int OFF_LC = TILE_END + (NH == 8 ? 16 : 0);             // [tokens][NH heads] f32 logit corrections of one group (32), or of a step of a longer one (64)
    static constexpr int LDS_WAVE = OFF_LC + (LONG ? 64 : 32) * NH * 4;      // 13376 (4 heads) / 14480 (8 heads), LONG 784 / 1296 more
    static_assert(OFF_KT % 16 == 0 && OFF_PT % 16 == 0 && OFF_VZ % 16 == 0 && OFF_TILE % 16 == 0 && OFF_LC % 16 == 0, "b128 alignment");
    static_assert(OFF_KT - KT_ROW >= OFF_ZERO, "code row -1: the constant rows");
    static_assert(OFF_TILE - TILE_ROW >= OFF_ZPP + 512, "tile row -1: behind what is staged for K");
    static_assert(OFF_LC - NH * 4 >= TILE_END - (TILE_ROW - 256), "corrections of row -1: behind the tile's last channel");
};
// LDS is handed out in pieces of 1280 bytes (768 workgroups of 53760 bytes on 256 compute units take one round, of 53776 two).
// Longer groups (56640 bytes, and more than 168 registers) have two workgroups a compute unit, not three.
constexpr int lds_of(int workgroup_bytes) { return (workgroup_bytes + 1279) / 1280 * 1280; }
// Workgroups resident on a compute unit, by registers and LDS; the launcher deals out as many shares (`lean` in ommx_host.cpp).
constexpr int resident(int nh, bool longer) { return nh == 4 && !longer ? OMMX_GQA4_WAVES : 2; }
static_assert(resident(4, false) * lds_of(4 * LdsMap<4, false>::LDS_WAVE) <= 160 * 1024, "4 heads, 32-token groups");
static_assert(resident(4, true) * lds_of(4 * LdsMap<4, true>::LDS_WAVE) <= 160 * 1024, "4 heads, longer groups");
static_assert(resident(8, true) * lds_of(4 * LdsMap<8, true>::LDS_WAVE) <= 160 * 1024, "8 heads");

// The running maximum of the online softmax is refreshed when a logit (base 2) exceeds it by this.  Under a maximum that lags,
// the largest weight is no longer 1 but a number rounded to f16, and the lse takes over its rounding error (up to 2^-12).  Longer
// groups are refreshed at once, as on the kernel that served them before: one split over 6001 tokens of 64 x 64 vectors, error of
// the lse 3.5e-5 there, 1.07e-4 with a slack of 8 (rms), of the output 6.4e-5 and 8.1e-5 (2-norm).
template <bool LONG>
constexpr float MAX_SLACK = LONG ? 0.0f : 8.0f;
// Longer groups were served before by a kernel with bf16 operands for K, which hold every step, and steps of V down to 2^-24.
// They keep that range.  A wave that meets a step of K or V outside 2^-14..2^15 (normal f16 numbers) with a code that is not
// zero, or a zero point of K from 2^18 on, or that has a query of 2^12 or more, drops what it has and walks its split in a
// second form (ANY): K codes and zero points as bf16, V codes times a step that may be subnormal, neither with a constant to
// take out again, and outlier entries that no normal f16 holds settled exactly.  (V steps above 2^15 stay held and
// reported.)  Steps that do not matter, of channels and rows that do not vary, stay in the first form (up to 9 % slower).
// Whole call over a kernel without any of it 0.99 to 0.98; the same as branches of the one loop 0.96 to 0.92, as a second loop that
// took over in the middle, with the sums so far, 0.99 to 0.93.  The looks go where the loop has a branch already: one
// of its own where V is staged cost 4 to 8 %.
constexpr int MIN_STEP_EXP = -14;
constexpr uint16_t ANY_ZP_BF16 = 0x4880u;           // 2^18: over 4, the smallest A scale, it is past the largest f16
constexpr float MAX_F16 = 65504.0f;
// Below the smallest normal f16 an entry is rounded to 2^-25 whatever its size, which a query of 2^12 and more (one that was
// divided by 2^HUGE_Q_DOWN) makes 1.7e-4 of a logit: the residual of such entries is added too.
constexpr float MIN_F16 = 6.103515625e-5f;
constexpr int HUGE_Q_DOWN = 6;

// K pair p of a code dword: channels p (low half) and p+8 (high half) as f16 with the 2-bit
// code at mantissa bits [2m+1:2m], m = k_pos(p), where the element reads
// (1 + code * 2^(2m-10)) * 2^e; the A operand of that channel carries q * 2^(10-2m).  Positions 2..4, so that
// only pairs 0, 1 (up four bits) and 5..7 (down six) need a shift; m = 1 (pair 1 unshifted) would carry a constant
// four times as large through the sums, and the error of the logits with it.  Longer groups have larger steps and
// fewer roundings elsewhere (their outliers are often exact): they take positions 3 and 4, two more shifts a dword.
template <bool LONG>
__host__ __device__ constexpr int k_pos(int p) {
    if (LONG) return p <= 1 ? p + 3 : p == 2 ? 3 : p <= 4 ? p : p == 5 ? 3 : 4;
    return p <= 1 ? p + 2 : (p <= 4 ? p : p - 3);
}
template <int P, bool LONG>
__device__ __forceinline__ uint32_t k_pair(uint32_t w, uint32_t w_up, uint32_t w_dn6, uint32_t magic) {
    const uint32_t sh = LONG ? (P <= 1 ? w_up : P == 2 ? w << 2 : P <= 4 ? w : P <= 6 ? w >> 4 : w_dn6)
                             : (P <= 1 ? w_up : P <= 4 ? w : w_dn6);
    return (sh & (0x00030003u << (2 * k_pos<LONG>(P)))) | magic;
}
// V channel y of a merged dword (token a in the low 16 bits, token b in the high 16 bits) as
// f16 (1 + c/16) * 2^e (even y, code at mantissa bits [7:6]) or (1 + c/4) * 2^e (odd y, bits
// [9:8]); `step` holds the f16 2^e of the two tokens.  The epilogue takes the constant out of the sum and multiplies what is
// left by 16 or 4, the fp32 sum's own rounding with it: longer groups take bits [9:8] for every channel (three more shifts a
// dword), without which one split over 16 K tokens of 64 x 64 vectors came out 1.22 times as far from 64-bit sums as the
// kernel that served them before.
template <int Y, bool LONG>
__device__ __forceinline__ uint32_t v_pair(uint32_t m, uint32_t step) {
    if constexpr (LONG) return ((Y <= 4 ? m << (8 - 2 * Y) : m >> (2 * Y - 8)) & 0x03000300u) | step;
    const uint32_t sh = Y <= 1 ? (m << 6) : Y <= 3 ? (m << 2) : Y <= 5 ? (m >> 2) : (m >> 6);
    return (sh & ((Y & 1) ? 0x03000300u : 0x00C000C0u)) | step;
}
// The same without its constant (ANY): code / 4 * 2^e, the step possibly subnormal.
template <int Y, bool LONG, bool ANY>
__device__ __forceinline__ uint32_t v_op(uint32_t m, uint32_t step) {
    if constexpr (!ANY) return v_pair<Y, LONG>(m, step);
    const f16x2 one = {1.0f, 1.0f};
    return __builtin_bit_cast(uint32_t, (__builtin_bit_cast(f16x2, v_pair<Y, LONG>(m, 0x3C003C00u)) - one) * __builtin_bit_cast(f16x2, step));
}
__device__ __forceinline__ uint32_t pk_u16(uint32_t lo, uint32_t hi) { return (lo & 0xFFFFu) | (hi << 16); }

// IDX: 0 = outlier positions from 32-bit bitmaps, 1 = from 7-bit position streams.
// OWN_MAP: outliers decode through their own (map_scale, centre) pair; false = through the
// base scale and zero point.  PARTIAL: the kv head serves 1 or 2 q heads (spare head slots repeat
// the last head and are not written).  ORDER: 0 one request, 1 up to 64 requests served longest
// first, 2 up to 256 (radix select); see ommx_decode.hip.
// NH: q heads per kv head the matrix rows and columns are laid out for, 4 or 8.
// GEN: the general form of the recipe: 1..8 outliers per vector (a.kout, bitmap plane only), and
// head_dim 64 (a.half, or HALF when nothing else is general): the planes of two neighbouring 64-channel kv heads read exactly like one
// 128-channel head, so a wave takes the pair as one head whose q heads are those of both, each
// zero on the other one's channels, and writes each q head only its own half of the output.
// GTS: K groups of 32 << GTS tokens (position streams; V vectors then 32, 64 or 128 channels wide), 6 outliers, or
// 10 with 128 tokens (KSLOTS).  The 64 tokens of a step lie in one group then, whose parameters are held once and whose
// outliers are walked once a step; either half scatters all of them, the ones that lie elsewhere to a row of the tile
// that nobody reads, which costs their instructions (10 outliers per 128 tokens walked twice are 20 a step and channel,
// against 12 in a 32-token recipe) but no branch.  The work is dealt out in those 64-token steps:
// whole groups of 128 left a batch of 342 groups on 172 of 256 resident workgroups, four serial steps each.  Whole
// call, ommx_decode.hip's kernel on whole groups -> this one: 128 tokens and 10 outliers, 4 requests of 2 to 20 K
// 46.0 -> 28.9 us, one of 64 K 47.5 -> 35.2, 32 of 1 to 16 K 165 -> 113; 64 tokens and 6 outliers, 64 K 37.3 -> 30.6, 700 tokens
// 14.6 -> 10.9, 32 of 1 to 16 K 128 -> 99.
// Longer groups: a split that needs what f16 does not hold (MIN_STEP_EXP above), walked from its start; every output of the
// wave is written here then.
template <int ORDER, bool OWN_MAP, int NH, int KSLOTS, int GTS>
__device__ __forceinline__ void other_form() {
    // (the kernel's arguments, read again: kept for this they would take the scalar registers of the loop)
    const DecodeArgs& a = *(const DecodeArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    constexpr int IDX = 1;
    constexpr bool PARTIAL = false, GEN = false, HALF = false, ANY = true;
    {
#include "ommx_decode_gqa4_walk.h"
    }
other_form:;
}

template <int IDX, bool OWN_MAP, bool PARTIAL, int ORDER, int NH = 4, bool GEN = false, int KSLOTS = 6, int GTS = 0, bool HALF = false>
__global__ void __launch_bounds__(256, (GEN && KSLOTS == 8) ? 2 : resident(NH, GTS > 0)) decode_gqa4_kernel(DecodeArgs a) {
    constexpr bool ANY = false;
    {
#include "ommx_decode_gqa4_walk.h"
        return;
    }
other_form:
    if constexpr (GTS > 0) other_form<ORDER, OWN_MAP, NH, KSLOTS, GTS>();
}

}  // namespace

// Returns 0 when launched, 1 when the shape belongs to another kernel.
int OMMX_GQA4_LAUNCH(const DecodeArgs& a_in, int Dh, int R, const DecodeTail* tail, hipStream_t st) {
    DecodeArgs a = a_in;
    a.half = 0;
    if (a.scale_bf16 || a.v_bf16) return 1;
    // K groups of 64 / 128 tokens with position streams: 6 outliers, or 10 of 128; V vectors of 32, 64 or 128 channels
    const bool longer = a.gt == 64 || a.gt == 128;
    if (longer) {
        if (a.idx_repr != 1 || !(a.kout == 6 || (a.kout == 10 && a.gt == 128)) || Dh != 128 || !(R == 4 || R == 8) ||
            !(a.gc == 32 || a.gc == 64 || a.gc == 128))
            return 1;
    } else if (a.gt != 32 || a.gc != 32 || a.kout < 1 || a.kout > 8) {
        return 1;
    }
    if ((reinterpret_cast<uintptr_t>(a.q) & 3) || (a.q_sb & 1) || (a.q_sh & 1)) return 1;
    int nh;                                   // q heads of a wave's (pair of) kv head(s)
    if (Dh == 128 && (R == 1 || R == 2 || R == 4 || R == 8)) {
        nh = R;
    } else if (Dh == 64 && (R == 1 || R == 2 || R == 4) && a.Hkv % 2 == 0) {
        a.half = 1;                           // two 64-channel kv heads read as one 128-channel head
        a.Hkv /= 2;
        nh = 2 * R;
    } else {
        return 1;
    }
    {
        // the kernel addresses a plane by 32-bit byte offsets: it takes planes whose extents are given and
        // below 4 GiB (code rows: pages * page size * kv heads * 32 B; the widest group plane has 9 B per channel)
        const uint64_t lim = 0xFFFFFF00ull;
        if (a.n_pages <= 0 || a.n_gslots <= 0) return 1;
        if (static_cast<uint64_t>(a.n_pages) * static_cast<uint64_t>(a.ps) >= (1ull << 24)) return 1;
        if (static_cast<uint64_t>(a.n_pages) * a.ps * a.Hkv * 32ull > lim) return 1;
        if (static_cast<uint64_t>(a.n_gslots) * a.Hkv * D * (longer ? 9ull : 6ull) > lim) return 1;
    }
    const bool general = a.half || (a.kout != 6 && !longer);
    if (general && a.idx_repr != 0) return 1;       // the general form reads bitmaps only
    const int waves = (a.Hkv % 4 == 0) ? 4 : ((a.Hkv % 2 == 0) ? 2 : 1);
    // shares: the orders below hold up to 64 requests (one per lane), or 256 (four)
    if (a.shares > 0 && a.B > (longer || (nh < 4 && !general) ? 64 : 256)) return 1;
    a.t_slices = 0;
    if (TAIL) {
        a.t = *tail;
        a.t_slices = kTailParts * (a.half ? 2 : 1) * a.B;
    }
    const dim3 grid = a.shares > 0 ? dim3(a.Hkv / waves, a.shares + a.t_slices) : dim3(a.S, a.Hkv / waves, a.B + (a.t_slices + a.S - 1) / a.S);
    const dim3 block(64 * waves);
    const size_t shm = (size_t)waves * (longer ? (nh == 8 ? LdsMap<8, true>::LDS_WAVE : LdsMap<4, true>::LDS_WAVE)
                                              : (nh == 8 ? LdsMap<8, false>::LDS_WAVE : LdsMap<4, false>::LDS_WAVE));
    const bool own_map = a.k_ms != nullptr;
    const int order = a.B == 1 ? 0 : (a.B > 64 && a.B <= 256 ? 2 : 1);
#define OMMX_GO(IDX, MAP, PART, ORD, NH, GEN) \
    hipLaunchKernelGGL((decode_gqa4_kernel<IDX, MAP, PART, ORD, NH, GEN>), grid, block, shm, st, a)
#define OMMX_GO_GEN(MAP, PART, NH)                                                                          \
    do {                                                                                                    \
        if (a.kout <= 4) hipLaunchKernelGGL((decode_gqa4_kernel<0, MAP, PART, 2, NH, true, 4>), grid, block, shm, st, a); \
        else if (a.kout <= 6) hipLaunchKernelGGL((decode_gqa4_kernel<0, MAP, PART, 2, NH, true, 6>), grid, block, shm, st, a); \
        else hipLaunchKernelGGL((decode_gqa4_kernel<0, MAP, PART, 2, NH, true, 8>), grid, block, shm, st, a);             \
    } while (0)
#define OMMX_GO_ORD(IDX, MAP, PART, NH)                              \
    do {                                                             \
        if (order == 0) OMMX_GO(IDX, MAP, PART, 0, NH, false);       \
        else if (order == 2) OMMX_GO(IDX, MAP, PART, 2, NH, false);  \
        else OMMX_GO(IDX, MAP, PART, 1, NH, false);                  \
    } while (0)
#define OMMX_GO_LONG(MAP, NH, KO, GTS)                                                                                         \
    do {                                                                                                                       \
        if (order == 0) hipLaunchKernelGGL((decode_gqa4_kernel<1, MAP, false, 0, NH, false, KO, GTS>), grid, block, shm, st, a); \
        else hipLaunchKernelGGL((decode_gqa4_kernel<1, MAP, false, 1, NH, false, KO, GTS>), grid, block, shm, st, a);            \
    } while (0)
    if (longer) {
        switch ((nh == 8 ? 8 : 0) | (own_map ? 4 : 0) | (a.gt == 64 ? 0 : a.kout == 6 ? 1 : 2)) {
            case 0: OMMX_GO_LONG(false, 4, 6, 1); break;
            case 1: OMMX_GO_LONG(false, 4, 6, 2); break;
            case 2: OMMX_GO_LONG(false, 4, 10, 2); break;
            case 4: OMMX_GO_LONG(true, 4, 6, 1); break;
            case 5: OMMX_GO_LONG(true, 4, 6, 2); break;
            case 6: OMMX_GO_LONG(true, 4, 10, 2); break;
            case 8: OMMX_GO_LONG(false, 8, 6, 1); break;
            case 9: OMMX_GO_LONG(false, 8, 6, 2); break;
            case 10: OMMX_GO_LONG(false, 8, 10, 2); break;
            case 12: OMMX_GO_LONG(true, 8, 6, 1); break;
            case 13: OMMX_GO_LONG(true, 8, 6, 2); break;
            default: OMMX_GO_LONG(true, 8, 10, 2); break;
        }
        return 0;
    }
    // head_dim 64 with 6 outliers, up to 64 requests: the same form with all of that known at compile time (the general
    // one walks one channel after the other, looks its slot count up and searches its share over 256 requests: 1 request of
    // 1 K 10.4 -> 8.8 us, 2 of 12 K 19.1 -> 17.1, 8 of 8 K 27.9 -> 25.1, kernel alone)
    if (a.half && a.kout == 6 && order < 2) {
#define OMMX_GO_HALF(MAP, PART, ORD, NH) \
    hipLaunchKernelGGL((decode_gqa4_kernel<0, MAP, PART, ORD, NH, false, 6, 0, true>), grid, block, shm, st, a)
        switch ((nh == 8 ? 4 : 0) | (order ? 2 : 0) | (own_map ? 1 : 0)) {
            case 0: OMMX_GO_HALF(false, true, 0, 4); break;
            case 1: OMMX_GO_HALF(true, true, 0, 4); break;
            case 2: OMMX_GO_HALF(false, true, 1, 4); break;
            case 3: OMMX_GO_HALF(true, true, 1, 4); break;
            case 4: OMMX_GO_HALF(false, false, 0, 8); break;
            case 5: OMMX_GO_HALF(true, false, 0, 8); break;
            case 6: OMMX_GO_HALF(false, false, 1, 8); break;
            default: OMMX_GO_HALF(true, false, 1, 8); break;
        }
#undef OMMX_GO_HALF
        return 0;
    }
    if (general) {
        // one instantiation per (outlier map, head layout): outlier count, head count and head_dim at run time
        if (nh == 8) { if (own_map) OMMX_GO_GEN(true, false, 8); else OMMX_GO_GEN(false, false, 8); }
        else { if (own_map) OMMX_GO_GEN(true, true, 4); else OMMX_GO_GEN(false, true, 4); }
        return 0;
    }
    switch ((nh == 8 ? 8 : 0) | (nh < 4 ? 4 : 0) | (a.idx_repr ? 2 : 0) | (own_map ? 1 : 0)) {
        case 0: OMMX_GO_ORD(0, false, false, 4); break;
        case 1: OMMX_GO_ORD(0, true, false, 4); break;
        case 2: OMMX_GO_ORD(1, false, false, 4); break;
        case 3: OMMX_GO_ORD(1, true, false, 4); break;
        case 4: OMMX_GO(0, false, true, 1, 4, false); break;
        case 5: OMMX_GO(0, true, true, 1, 4, false); break;
        case 6: OMMX_GO(1, false, true, 1, 4, false); break;
        case 7: OMMX_GO(1, true, true, 1, 4, false); break;
        case 8: OMMX_GO_ORD(0, false, false, 8); break;
        case 9: OMMX_GO_ORD(0, true, false, 8); break;
        case 10: OMMX_GO_ORD(1, false, false, 8); break;
        default: OMMX_GO_ORD(1, true, false, 8); break;
    }
#undef OMMX_GO
#undef OMMX_GO_GEN
#undef OMMX_GO_LONG
#undef OMMX_GO_ORD
    return 0;
}

}  // namespace ommx
