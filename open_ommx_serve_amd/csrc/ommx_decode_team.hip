// Split-KV decode kernel for short calls: the serving recipe (32-token / 32-channel vectors, six outliers, int8 exponents,
// INT2 V) with FOUR WAVES on one kv head of one split instead of one.  Same operator, operands and arithmetic as the kernel of
// ommx_decode_gqa4.hip (see there); what differs is who does what.
//
// What bounds it: a short call takes as long as the chain of one wave, a lone wave issues an instruction every five clocks, and 64 tokens x
// 128 channels are 886 vector instructions and a dozen LDS round trips (2.8 us for a lone 32-token group, 3.9 for two).  Here a workgroup
// is one kv head (head_dim 64: a pair of them) and each wave owns 32 of its channels, which is one V vector of a token and one MFMA
// k-step:
//   * channel pass: lane = (group, channel), so both groups of a step are walked at once, six outliers a lane instead of 24;
//   * QK: one base and one tile MFMA per 16 tokens on top of an accumulator that starts as the group's bias (sum q*zp - sum A*2^e);
//     the waves' partial logits meet in LDS (one barrier a step), where every wave adds them up in the same order;
//   * softmax: by every wave for itself, from the same numbers (a second exchange would cost more than the 40 instructions);
//   * P.V: two 16-channel blocks of the wave's own V vector.
// About a quarter more instructions in all, but a third as many in a chain: a step of two groups 1.6 us.  Of a call of 1 K tokens (15 splits
// of 8 heads, one step each) the walk takes 4 us -- arguments 0.6, length and tables together 0.5, rows 0.7, the step 1.6, the state 0.4 --,
// hand-over and merge 2.7.  Whole call, one wave a head and a merge of its own -> this: 1 K tokens 9.5 -> 8.2 us, 3 requests of 0.7 to
// 9 K with one kv head 12.1 -> 9.9, 2 x 12 K of 64 channels 18.3 -> 15.9, 6 K 13.9 -> 11.9, 8 K with 64 q heads 19.8 -> 16.6; a batch of
// eight served token by token 1.70 -> 1.42 ms for 80 steps of a layer.  38 to 53 KB of LDS a workgroup.
// (walk repeats the channel pass, QK, softmax and P.V of ommx_decode_gqa4_walk.h for 32 channels: a correction there is one here too.)
#include <type_traits>

#include "ommx_decode_recipe.h"
#include "ommx_decode_shares.h"
#include "ommx_decode_tail.h"

namespace ommx {

namespace {

using namespace decode_util;

constexpr int WAVES = 4;                 // of a workgroup; 32 channels each
constexpr int D = 128;                   // channels of a workgroup: a kv head, or a pair of 64-channel ones
constexpr int KT_ROW = 8;                // bytes of a staged K code row: the wave's 32 channels
constexpr int TILE_ROW = 80;             // bytes per row of the outlier tile (64 used): 16 rows read as b128 spread over all banks
constexpr int TILE_GROUP = 33;           // rows of a group: one that nobody reads (position -1, see lowest_bit), then its 32 tokens
constexpr int VT_COL = 68;               // dwords per V dword column (64 used)
constexpr int PT_ROW = 72;               // halfwords per row of the f16 [row][64 tokens] arrays

// LDS of a workgroup: constants, the exchange of partial logits (two steps' worth, so that one barrier a step is enough),
// then a region per wave.
// FINE: outliers decode through the base scale.  Their entries are exact then, and the f16 rounding of the softmax weights is what is
// left of the error: it is settled by a second f16 (splits of 64 tokens instead of 32, of which only the largest weight is exact, would
// make it 1.3 times what it was).
template <int NH, bool FINE>
struct TeamLds {
    static constexpr int OFF_ZERO = 0;                              // 128 B of zeros
    static constexpr int OFF_ONES = 128;                            // 128 B of f16 1.0
    static constexpr int OFF_X = 256;                               // [2][WAVES][64 tokens][NH] f32
    static constexpr int X_WAVE = 64 * NH * 4, X_STEP = WAVES * X_WAVE;
    static constexpr int OFF_WAVES = OFF_X + 2 * X_STEP;
    // of a wave
    static constexpr int OFF_KT = 0;                                // [64 tokens] K code rows
    static constexpr int OFF_MAG = OFF_KT + 64 * KT_ROW;            // [2 groups][32] f16 2^e, pair order
    static constexpr int OFF_ZPP = OFF_MAG + 128;                   // same order, f16 zero points over the A scale
    static constexpr int OFF_VT = OFF_ZPP + 128;                    // [2 dword columns][VT_COL]
    static constexpr int OFF_PT = OFF_VT + 2 * VT_COL * 4;          // [NH][PT_ROW] f16 softmax weights
    static constexpr int OFF_PL = OFF_PT + NH * PT_ROW * 2;         // FINE: what the weights' rounding dropped, the same again
    static constexpr int OFF_VZ = OFF_PL + (FINE ? NH * PT_ROW * 2 : 0);     // [PT_ROW] f16 V zero points
    static constexpr int OFF_VS = OFF_VZ + PT_ROW * 2;              // [PT_ROW] f16 2^e_v
    static constexpr int OFF_TILE = OFF_VS + PT_ROW * 2;            // [2][TILE_GROUP][TILE_ROW] f16 outlier entries
    static constexpr int LDS_WAVE = OFF_TILE + 2 * TILE_GROUP * TILE_ROW;
    static constexpr int BYTES = OFF_WAVES + WAVES * LDS_WAVE;      // 38272 (4 heads) / 48768 (8), FINE 40576 / 53376
    static_assert(OFF_PT % 16 == 0 && OFF_VZ % 16 == 0 && OFF_TILE % 16 == 0 && LDS_WAVE % 16 == 0, "b128 alignment");
    static_assert(LDS_WAVE >= (32 * NH + 2 * NH) * 4, "the tail rows' share of it");
};
// Workgroups a compute unit holds (LDS in pieces of 1280 bytes): the register budget is set for them.
constexpr int team_resident(int nh) { return nh == 4 ? 3 : 2; }
static_assert(team_resident(4) * ((TeamLds<4, true>::BYTES + 1279) / 1280 * 1280) <= 160 * 1024, "4 heads");
static_assert(team_resident(8) * ((TeamLds<8, true>::BYTES + 1279) / 1280 * 1280) <= 160 * 1024, "8 heads");

// All waves of the workgroup: what they wrote to LDS before is there for all of them after.  (Loads from memory stay under way.)
__device__ __forceinline__ void team_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// What the kernel needs of a call, strides as 32-bit numbers (the launcher sees to it that everything they reach lies within
// 2^32 bytes): the scalar arithmetic of addresses is a quarter of a short call's instructions.
struct TeamArgs {
    // the merge: as in TeamMerge
    unsigned long long* arrivals; uint64_t number;
    float* o; uint16_t* o16; float* lse;
    int64_t o_b, o_h, lse_b;
    const int32_t* seq;
    const uint16_t* q;
    const uint8_t* k_base; const int8_t* k_scale; const uint16_t* k_zp; const uint16_t* k_ms; const uint16_t* k_mc;
    const uint8_t* k_obmp; const uint8_t* k_oval; const uint8_t* v_main; const int8_t* v_scale; const uint16_t* v_zp;
    const char* rt; const char* rg;
    float* al; float* sl;
    int32_t* err;
    uint32_t rt_b, rg_b;                     // bytes between the table rows of two requests
    int rt_n, rg_n;                          // entries of a table row
    uint32_t q_sb, q_sh, al_b, al_h, al_s, sl_b, sl_h, sl_s;
    int heads, Hkv;                          // q heads of a workgroup; workgroups across (kv heads, or pairs of them)
    int ps_sh, tsh, tok_off, n_pages, n_gslots;
    int S, per;                              // splits of a request and groups in each (fixed), or the most shares of one
    float sm_scale, cap;
    int B, shares, shares_few, singles;
    int32_t* share_count;
    int tails;                               // workgroups of a kv head (HALF: of a pair) that attend its tail rows; 0 without any
    DecodeTail t;
};
// The kernel's arguments read again from where they lie, for parts that come late or that only some workgroups run: kept for
// them, the arguments would take the scalar registers of the walk (a hundred spills, 1.5 us of a short call).
__device__ __forceinline__ const TeamArgs& args_again() {
    auto p = (const __attribute__((address_space(4))) TeamArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const TeamArgs*)p;
}

// Position m of a channel's code in the mantissa, as k_pos in ommx_decode_gqa4.hip: 2 for even channels, 3 for odd ones.
// The A operand of the channel carries q * 2^(10-2m), what is added to its base code 2^-(10-2m).
__device__ __forceinline__ uint32_t k_or(uint32_t w, uint32_t mask, uint32_t step) { return (w & mask) | step; }

// The walk of one split: groups [g_first, g_first + g_count) of request b, at least one.  `page`, `slot`: tables of its first step as
// fetch_tables left them, if `tables` says that they have been asked for.
template <int IDX, bool OWN_MAP, int NH, bool HALF>
__device__ __forceinline__ void walk(const TeamArgs& a, uint8_t* const smem, int unit, int b, int L, uint32_t sp, uint32_t g_first, uint32_t g_count,
                                     int page, int slot, bool tables, int lane, int wave) {
    constexpr bool FINE = !OWN_MAP;
    using Lds = TeamLds<NH, FINE>;
    uint8_t* const sm = smem + Lds::OFF_WAVES + wave * Lds::LDS_WAVE;
    const int j = lane & 15, kq = lane >> 4;
    const int heads = a.heads, R = HALF ? heads >> 1 : heads;             // q heads of the wave's kv head
    const int qh0 = unit * heads + (HALF ? (wave >> 1) * R : 0);
    const int ch0 = HALF ? 32 * (wave & 1) : 32 * wave;                   // first of the wave's channels in its head
    const int g = lane >> 5, c = lane & 31;                               // channel pass: lane = (group of the step, channel)
    // q: this lane's 8 channels of head j % NH (A operand), and channel c of every head (thresholds)
    uint32_t qw[4];
    uint16_t qc[NH];
    {
        // (a scalar base and 32-bit lane offsets)
        const char* const qb = reinterpret_cast<const char*>(a.q) + 2u * (b * a.q_sb + qh0 * a.q_sh + ch0);
        const uint32_t q_sh = 2u * a.q_sh;
        const uint32_t qh = __umul24(static_cast<uint32_t>(min(j & (NH - 1), R - 1)), q_sh) + 32 * (kq & 1) + 8 * (kq >> 1);
#pragma unroll
        for (int i = 0; i < 4; ++i) qw[i] = *reinterpret_cast<const uint32_t*>(qb + (qh + 16 * (i >> 1) + 4 * (i & 1)));
#pragma unroll
        for (int r = 0; r < NH; ++r) qc[r] = *reinterpret_cast<const uint16_t*>(qb + min(r, R - 1) * q_sh + 2u * c);
    }
    const int n_begin = static_cast<int>(g_first << 5), n_end = min(static_cast<int>((g_first + g_count) << 5), L);
    // ---- addressing: scalar plane pointers and 32-bit byte offsets, as in ommx_decode_gqa4.hip ------------------
    const uint32_t Hk = static_cast<uint32_t>(a.Hkv), row_bytes = Hk * 32u;
    const int last = n_end - 1, tok_off = a.tok_off, ps_sh = a.ps_sh, tsh = a.tsh;
    const char* const rt_b = a.rt + b * a.rt_b;
    const char* const rg_b = a.rg + b * a.rg_b;
    const int part = 4 * unit + wave;                                     // V vector and 8-byte piece of a code row
    const uint8_t* const kb = a.k_base + 8 * part;
    const uint8_t* const vb = a.v_main + 8 * part;
    const int8_t* const vs = a.v_scale + part;
    const uint16_t* const vz = a.v_zp + part;
    auto at = [](const void* base, uint32_t byte_off) { return static_cast<const char*>(base) + byte_off; };
    bool bad_id = false, over_step = false;
    auto fetch_tables = [&](int n) {
        page = *reinterpret_cast<const int*>(rt_b + ((uint32_t)((min(n + lane, last) + tok_off) >> ps_sh) << tsh));
        slot = *reinterpret_cast<const int*>(rg_b + ((uint32_t)min((n >> 5) + g, last >> 5) << tsh));
    };
    u32x2 kr, vr;
    uint32_t row = 0, vsc, vzp;
    auto fetch_k = [&](int n) {
        page = clamp_id(page, a.n_pages, bad_id);
        const int p = min(n + lane, last) + tok_off;
        row = __umul24(static_cast<uint32_t>((page << ps_sh) + (p & ((1 << ps_sh) - 1))), row_bytes);
        kr = *reinterpret_cast<const u32x2*>(at(kb, row));
    };
    auto fetch_v = [&]() {
        vr = *reinterpret_cast<const u32x2*>(at(vb, row));
        vsc = *reinterpret_cast<const uint8_t*>(at(vs, row >> 3));
        vzp = *reinterpret_cast<const uint16_t*>(at(vz, row >> 2));
    };
    uint32_t g_sc, g_zp, g_ms = 0, g_mc = 0, g_ix0, g_ix1 = 0, g_ov0, g_ov1;
    auto fetch_params = [&]() {
        const uint32_t ch = (static_cast<uint32_t>(clamp_id(slot, a.n_gslots, bad_id)) * Hk + unit) * D + 32u * wave + c;
        g_sc = *reinterpret_cast<const uint8_t*>(at(a.k_scale, ch));
        g_zp = *reinterpret_cast<const uint16_t*>(at(a.k_zp, 2 * ch));
        if (OWN_MAP) {
            g_ms = *reinterpret_cast<const uint16_t*>(at(a.k_ms, 2 * ch));
            g_mc = *reinterpret_cast<const uint16_t*>(at(a.k_mc, 2 * ch));
        }
        if (IDX == 0) {
            g_ix0 = *reinterpret_cast<const uint32_t*>(at(a.k_obmp, 4 * ch));
        } else {          // six bytes: of the two dwords that hold them the upper or the lower ones
            g_ix0 = *reinterpret_cast<const uint32_t*>(at(a.k_obmp, (6 * ch) & ~3u));
            g_ix1 = *reinterpret_cast<const uint32_t*>(at(a.k_obmp, ((6 * ch) & ~3u) + 4));
        }
        // three nibble bytes: the dwords of the first and of the last of them
        g_ov0 = *reinterpret_cast<const uint32_t*>(at(a.k_oval, (3 * ch) & ~3u));
        g_ov1 = *reinterpret_cast<const uint32_t*>(at(a.k_oval, (3 * ch + 2) & ~3u));
    };
    if (tables) {
        // asked for before the length was here: past the last token and the last group these again
        const int over = last - n_begin;
        const int last_page = __builtin_amdgcn_readlane(page, over & 63), first_slot = __builtin_amdgcn_readlane(slot, 0);
        if (lane > over) page = last_page;
        if (over < 32) slot = first_slot;
    } else {
        fetch_tables(n_begin);
    }
    asm volatile("" ::: "memory");
    // The largest |q| from 2^7 on: the query is taken divided by a power of two (ommx_decode_gqa4.hip), by each wave for its own
    // channels; its logits are multiplied by it again before they meet the others'.
    int q_down = 0;
    {
        float qa = 0.0f;
#pragma unroll
        for (int r = 0; r < NH; ++r) qa = fmaxf(qa, fabsf(__uint_as_float(static_cast<uint32_t>(qc[r]) << 16)));
        if (__builtin_expect(any_lane(qa >= 128.0f), 0)) {
            float m4[4] = {qa, qa, qa, qa};
            wave_max4(m4);
            q_down = min(static_cast<int>((__float_as_uint(m4[0]) >> 23) & 0xFFu) - 127 - 6, 100);
        }
    }
    const float q_mul = __uint_as_float(static_cast<uint32_t>(127 - q_down) << 23), q_back = __uint_as_float(static_cast<uint32_t>(127 + q_down) << 23);
    // ---- A operand: q * 2^(10-2m) of head j % NH, k = (kq, i) <-> channel 16 (kq & 1) + 4 (kq >> 1) + i / 2 + 8 (i % 2)
    u32x4 aq, aq_neg;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        auto q_at = [&](uint32_t w) { return __uint_as_float((r & 1) ? (w & 0xFFFF0000u) : (w << 16)); };
        const float qs = ((r & 1) ? 16.0f : 64.0f) * q_mul;
        aq[r] = pack_f16x2(qs * q_at(qw[r >> 1]), qs * q_at(qw[2 + (r >> 1)]));
        aq_neg[r] = aq[r] ^ 0x80008000u;
    }
    // rows first, the constants below while they are on their way
    fetch_k(n_begin);
    fetch_params();
    fetch_v();
    if (n_begin + 64 < n_end) fetch_tables(n_begin + 64);
    asm volatile("" ::: "memory");
    // where the state goes (worked out here, while the rows are on their way)
    const uint32_t al_h = 4u * a.al_h, sl_h = 4u * a.sl_h;
    char* const al = reinterpret_cast<char*>(a.al) + (b * 4u * a.al_b + qh0 * al_h + 4u * (sp * a.al_s + ch0));
    char* const sl = reinterpret_cast<char*>(a.sl) + (b * 4u * a.sl_b + qh0 * sl_h + 4u * (sp * a.sl_s));
    {
        u32x4* p = reinterpret_cast<u32x4*>(sm + Lds::OFF_TILE);
        constexpr int PIECES = 2 * TILE_GROUP * TILE_ROW / 16;
#pragma unroll
        for (int i = 0; i + 64 <= PIECES; i += 64) p[i + lane] = u32x4{0, 0, 0, 0};
        if (lane < PIECES % 64) p[PIECES / 64 * 64 + lane] = u32x4{0, 0, 0, 0};
        // (the constants are the workgroup's: every wave writes them, so that none has to wait for another)
        if (lane < 16) reinterpret_cast<u32x4*>(smem + Lds::OFF_ZERO)[lane] =
            lane < 8 ? u32x4{0, 0, 0, 0} : u32x4{0x3C003C00u, 0x3C003C00u, 0x3C003C00u, 0x3C003C00u};
    }
    f32x4 acc[2] = {f32x4{0, 0, 0, 0}, f32x4{0, 0, 0, 0}}, accz = {0, 0, 0, 0};
    float m_run[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) m_run[r] = -INFINITY;
    // ---- lane constants --------------------------------------------------------------------------------------
    const uint32_t y = c & 15;
    const uint32_t hw = 8 * ((c >> 4) + 2 * ((y & 7) >> 2)) + 2 * (y & 3) + (y >> 3);      // halfword of channel c in pair order
    const float cs = (c & 1) ? 1.0f / 16.0f : 1.0f / 64.0f;                                // 2^-(10-2m)
    const float sm_scale = a.sm_scale;
    float big_thr;                         // the |tile entry| from which its f16 rounding matters (infinite for q = 0)
    {
        float qm = 0.0f;
#pragma unroll
        for (int r = 0; r < NH; ++r) qm = fmaxf(qm, fabsf(__uint_as_float(static_cast<uint32_t>(qc[r]) << 16)) * q_mul);
        big_thr = (HALF ? 0.75f : 1.0f) * BIG_DELTA * 16.0f * BIG_DELTA_SM_SCALE * cs * __builtin_amdgcn_rcpf(qm * sm_scale * q_back);
    }
    const uint8_t* const kt_lane = sm + Lds::OFF_KT + 32 * KT_ROW * g + (c >> 2);          // the channel's code byte, row 0 of the group
    const uint32_t code_bits = 3u << (2 * (c & 3));
    const int code_unit = 24 - 2 * (c & 3);                                                // as in ommx_decode_gqa4.hip
    uint8_t* const tile_lane = sm + Lds::OFF_TILE + (TILE_GROUP * g + 1) * TILE_ROW + 2 * hw;
    const uint32_t nib_sh = 8u * ((3u * c) & 3u);
    const uint32_t w_sh = 8u * (kq >> 1);
    const float c2 = sm_scale * 1.4426950408889634f;
    uint32_t x_at = Lds::OFF_X;            // the step's exchange

    for (int n0 = n_begin; n0 < n_end; n0 += 64) {
        const bool more = n0 + 64 < n_end, g1_live = n0 + 32 < n_end;
        // ------------------------------------------------------------------ stage K
        int e = static_cast<int8_t>(g_sc);
        const bool exact_step = any_lane(e >= EXACT_STEP_EXP) || q_down != 0;
        if (__builtin_expect(exact_step, 0)) {
            over_step |= any_lane(e > MAX_STEP_EXP);
            e = min(e, CODE_STEP_EXP);
        }
        const float zp = __uint_as_float(g_zp << 16);
        *reinterpret_cast<u32x2*>(sm + Lds::OFF_KT + KT_ROW * lane) = kr;
        reinterpret_cast<uint16_t*>(sm + Lds::OFF_MAG)[32 * g + hw] =
            static_cast<uint16_t>((min(max(e, -15), MAX_STEP_EXP) + 15) << 10);
        reinterpret_cast<uint16_t*>(sm + Lds::OFF_ZPP)[32 * g + hw] = static_cast<uint16_t>(pack_f16x2(cs * zp, 0.0f));
        lds_fence();
        if (more) fetch_k(n0 + 64);
        // ------------------------------------------------------------------ channel pass (ommx_decode_gqa4.hip, walk_read / walk_write)
        bool res_any;
        int pos[6];
        float dls[6];
        {
            uint32_t cb[6];
            uint32_t bm = g_ix0;
            uint32_t ix_lo = 0, ix_hi = 0;
            if (IDX == 1) {
                ix_lo = (c & 1) ? __builtin_amdgcn_alignbit(g_ix1, g_ix0, 16) : g_ix0;
                ix_hi = (c & 1) ? g_ix1 >> 16 : g_ix1;
            }
#pragma unroll
            for (int s = 0; s < 6; ++s) {
                if (IDX == 0) {
                    pos[s] = lowest_bit(bm);
                    if (s < 5) bm = without_bit(bm, pos[s]);
                } else {
                    pos[s] = s < 4 ? ((ix_lo >> (7 * s)) & 31) : s == 4 ? (__builtin_amdgcn_alignbit(ix_hi, ix_lo, 28) & 31) : ((ix_hi >> 3) & 31);
                }
                cb[s] = kt_lane[pos[s] * KT_ROW];
            }
            const float code_step = __builtin_ldexpf(cs, e + code_unit);
            float a1, b1;
            if (OWN_MAP) {
                a1 = cs * __builtin_amdgcn_rcpf(__uint_as_float(g_ms << 16));
                b1 = cs * (__uint_as_float(g_mc << 16) - zp);
            } else {
                a1 = __builtin_ldexpf(cs, e);
                b1 = 0.0f;
            }
            const uint32_t nib = __builtin_amdgcn_alignbit(g_ov1, g_ov0, nib_sh);
            const f32x2 l01 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(nib, 1.0f, 0), l23 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(nib, 1.0f, 1),
                        l45 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(nib, 1.0f, 2);
            const float lv[6] = {l01[0], l01[1], l23[0], l23[1], l45[0], l45[1]};
            float dl_max = 0.0f;
#pragma unroll
            for (int s = 0; s < 6; ++s) {
                float dl = fmaf(-f16_bits(cb[s] & code_bits), code_step, fmaf(lv[s], a1, b1));
                // (the entry as a value of its own: rounded to f16 here exactly as below)
                asm("" : "+v"(dl));
                dls[s] = dl;
                *reinterpret_cast<uint16_t*>(tile_lane + pos[s] * TILE_ROW) = __builtin_bit_cast(uint16_t, static_cast<_Float16>(dl));
                dl_max = fmaxf(dl_max, fabsf(dl));
            }
            res_any = any_lane(dl_max >= big_thr);
        }
        lds_fence();
        if (more) fetch_params();
        // ------------------------------------------------------------------ QK
        f32x4 d[4];
        u32x4 mag[2];
        const u32x4 none = {0, 0, 0, 0};
        u32x4* const tile_row = reinterpret_cast<u32x4*>(sm + Lds::OFF_TILE + (1 + j) * TILE_ROW + 16 * kq);
        constexpr int BLOCK = 16 * TILE_ROW / 16, GROUP = TILE_GROUP * TILE_ROW / 16;
        // EX: the operand without its constant, for large steps (EXACT_STEP_EXP)
        auto qk = [&](auto EX, auto GROUPS) {
            constexpr int NB = 2 * decltype(GROUPS)::value;
            u32x4 bt[4];
            uint32_t w[4];
            f32x4 bias[2];
#pragma unroll
            for (int gg = 0; gg < NB / 2; ++gg) {       // (the same zero points and steps for every column)
                const u32x4 zpp = *reinterpret_cast<const u32x4*>(sm + Lds::OFF_ZPP + 64 * gg + 16 * kq);
                mag[gg] = *reinterpret_cast<const u32x4*>(sm + Lds::OFF_MAG + 64 * gg + 16 * kq);
                bias[gg] = mfma_f16(aq, zpp, f32x4{0, 0, 0, 0});
            }
#pragma unroll
            for (int t = 0; t < NB; ++t) bt[t] = tile_row[(t >> 1) * GROUP + (t & 1) * BLOCK];
#pragma unroll
            for (int t = 0; t < NB; ++t) tile_row[(t >> 1) * GROUP + (t & 1) * BLOCK] = none;
#pragma unroll
            for (int t = 0; t < NB; ++t)
                w[t] = *reinterpret_cast<const uint32_t*>(sm + Lds::OFF_KT + (16 * t + j) * KT_ROW + 4 * (kq & 1)) >> w_sh;
            if constexpr (!decltype(EX)::value) {
#pragma unroll
                for (int gg = 0; gg < NB / 2; ++gg) bias[gg] = mfma_f16(aq_neg, mag[gg], bias[gg]);
            }
            // (the constants of the base codes and of the bias cancel before the entries are added: on top of them these lost bits,
            // 1.3 times the error where outliers have no map of their own)
#pragma unroll
            for (int t = 0; t < NB; ++t) {
                const u32x4 mg = mag[t >> 1];
                uint32_t op[4] = {k_or(w[t] << 4, 0x00300030u, mg[0]), k_or(w[t] << 4, 0x00C000C0u, mg[1]),
                                  k_or(w[t], 0x00300030u, mg[2]), k_or(w[t], 0x00C000C0u, mg[3])};
                if constexpr (decltype(EX)::value) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const uint32_t step = mg[r];
                        op[r] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, op[r]) - __builtin_bit_cast(f16x2, step));
                    }
                }
                d[t] = mfma_f16(aq, u32x4{op[0], op[1], op[2], op[3]}, bias[t >> 1]);
            }
#pragma unroll
            for (int t = 0; t < NB; ++t) d[t] = mfma_f16(aq, bt[t], d[t]);
        };
        d[2] = d[3] = f32x4{0, 0, 0, 0};
        if (__builtin_expect(exact_step, 0)) {
            if (g1_live) qk(std::true_type{}, std::integral_constant<int, 2>{});
            else qk(std::true_type{}, std::integral_constant<int, 1>{});
        } else if (g1_live) {
            qk(std::false_type{}, std::integral_constant<int, 2>{});
        } else {
            qk(std::false_type{}, std::integral_constant<int, 1>{});
        }
        // Some entry's f16 rounding matters: what it dropped goes through the tile as well (another 11 bits; one entry on most steps'
        // logits.  As float atomics on the logits, head by head: 650 clocks instead of 300, with the other waves waiting)
        if (res_any) {
            lds_fence();
#pragma unroll
            for (int s = 0; s < 6; ++s)
                *reinterpret_cast<uint16_t*>(tile_lane + pos[s] * TILE_ROW) = __builtin_bit_cast(
                    uint16_t, static_cast<_Float16>(dls[s] - static_cast<float>(static_cast<_Float16>(dls[s]))));
            lds_fence();
            u32x4 bt[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) bt[t] = tile_row[(t >> 1) * GROUP + (t & 1) * BLOCK];
#pragma unroll
            for (int t = 0; t < 4; ++t) tile_row[(t >> 1) * GROUP + (t & 1) * BLOCK] = none;
#pragma unroll
            for (int t = 0; t < 4; ++t) d[t] = mfma_f16(aq, bt[t], d[t]);
        }
        // ------------------------------------------------------------------ partial logits
        // 4 heads: the lane keeps those of token n0 + lane; 8 heads: heads 4 (kq & 1)..+3 of tokens 16 (kq >> 1) + j of either group
        f32x4 part_x[NH / 4];
        if constexpr (NH == 4) {
            part_x[0] = (kq & 2) ? ((kq & 1) ? d[3] : d[2]) : ((kq & 1) ? d[1] : d[0]);
        } else {
            part_x[0] = (kq >> 1) ? d[1] : d[0];
            part_x[1] = (kq >> 1) ? d[3] : d[2];
        }
        const uint32_t x_lane = NH == 4 ? 16u * lane : 32u * (16u * (kq >> 1) + j) + 16u * (kq & 1);
#pragma unroll
        for (int i = 0; i < NH / 4; ++i) {
            f32x4* const xp = reinterpret_cast<f32x4*>(smem + x_at + wave * Lds::X_WAVE + x_lane + 1024 * i);
            if (__builtin_expect(q_down != 0, 0)) part_x[i] *= q_back;
            *xp = part_x[i];
        }
        if (more) fetch_tables(n0 + 128);
        // ------------------------------------------------------------------ stage V
        {
            uint32_t* const vt = reinterpret_cast<uint32_t*>(sm + Lds::OFF_VT) + lane;
            vt[0] = vr[0];
            vt[VT_COL] = vr[1];
            const int ev = static_cast<int8_t>(vsc);
            if (__builtin_expect(any_lane(ev > MAX_STEP_EXP), 0)) over_step = true;
            reinterpret_cast<uint16_t*>(sm + Lds::OFF_VS)[lane] = static_cast<uint16_t>((min(max(ev, -15), MAX_STEP_EXP) + 15) << 10);
            reinterpret_cast<uint16_t*>(sm + Lds::OFF_VZ)[lane] = static_cast<uint16_t>(pack_f16x2(__uint_as_float(vzp << 16), 0.0f));
        }
        if (more) fetch_v();
        team_barrier();
        // ------------------------------------------------------------------ softmax (ommx_decode_gqa4.hip)
        f32x4 xs[NH / 4];
#pragma unroll
        for (int i = 0; i < NH / 4; ++i) {
            const uint8_t* const xp = smem + x_at + (HALF ? (wave & 2) * Lds::X_WAVE : 0) + x_lane + 1024 * i;
            f32x4 v[HALF ? 2 : WAVES];
#pragma unroll
            for (int w = 0; w < (HALF ? 2 : WAVES); ++w) v[w] = *reinterpret_cast<const f32x4*>(xp + w * Lds::X_WAVE);
            xs[i] = HALF ? v[0] + v[1] : (v[0] + v[1]) + (v[HALF ? 0 : 2] + v[HALF ? 1 : 3]);
        }
        x_at ^= Lds::OFF_X ^ (Lds::OFF_X + Lds::X_STEP);
        if (a.cap > 0.0f) {
#pragma unroll
            for (int i = 0; i < NH / 4; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) xs[i][r] = apply_cap(xs[i][r] * sm_scale, a.cap) * 1.4426950408889634f;
        } else {
#pragma unroll
            for (int i = 0; i < NH / 4; ++i) xs[i] *= c2;
        }
        const int tk = NH == 4 ? lane : 16 * (kq >> 1) + j;
        if (n0 + 64 > n_end) {
#pragma unroll
            for (int i = 0; i < NH / 4; ++i)
                if (n0 + 32 * i + tk >= n_end) xs[i] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
        }
        float over = -INFINITY;
#pragma unroll
        for (int i = 0; i < NH / 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) over = fmaxf(over, xs[i][r] - m_run[r]);
        if (any_lane(over > 8.0f)) {        // the slack of ommx_decode_gqa4.hip's 32-token recipes
            float mxs[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) mxs[r] = NH == 4 ? xs[0][r] : fmaxf(xs[0][r], xs[NH / 4 - 1][r]);
            if constexpr (NH == 4) wave_max4(mxs);
            else rowpair_max4(mxs);
            float alpha[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float m_new = fmaxf(m_run[r], mxs[r]);
                alpha[r] = (m_run[r] == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(m_run[r] - m_new);
                m_run[r] = m_new;
            }
            // accumulators hold column (replica, head j % NH) in every register
            float al = (j & 3) == 0 ? alpha[0] : ((j & 3) == 1 ? alpha[1] : ((j & 3) == 2 ? alpha[2] : alpha[3]));
            if constexpr (NH == 8) {
                const float al_nb = lane_value(al, lane ^ 16);
                al = (((j >> 2) & 1) == (kq & 1)) ? al : al_nb;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) { acc[0][i] *= al; acc[1][i] *= al; accz[i] *= al; }
        }
        {
            _Float16* const pt = reinterpret_cast<_Float16*>(sm + Lds::OFF_PT) + (NH == 4 ? 0 : 4 * (kq & 1) * PT_ROW) + tk;
#pragma unroll
            for (int i = 0; i < NH / 4; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float w = __builtin_amdgcn_exp2f(xs[i][r] - m_run[r]);
                    const _Float16 w16 = static_cast<_Float16>(w);
                    pt[32 * i + r * PT_ROW] = w16;
                    if constexpr (FINE) pt[(Lds::OFF_PL - Lds::OFF_PT) / 2 + 32 * i + r * PT_ROW] = static_cast<_Float16>(w - static_cast<float>(w16));
                }
        }
        lds_fence();
        // ------------------------------------------------------------------ P.V (transposed)
        // Row i of the V operand is channel 16 (i >> 3) + 8 (i >> 2 & 1) + 4 a + (i & 3) of block a, its code at mantissa bits
        // [9:8]; rows of the sums operand: zero points, steps, ones.
        const uint32_t vsel = (j & 4) ? 0x07060302u : 0x05040100u;
        const uint8_t* const azp = j == 0 ? sm + Lds::OFF_VZ + 16 * kq : j == 1 ? sm + Lds::OFF_VS + 16 * kq
                                                                               : smem + (j == 2 ? Lds::OFF_ONES : Lds::OFF_ZERO) + 16 * kq;
#pragma unroll
        for (int kb2 = 0; kb2 < 2; ++kb2) {
            if (kb2 == 1 && !g1_live) break;
            const u32x4 pw = *reinterpret_cast<const u32x4*>(sm + Lds::OFF_PT + ((j & (NH - 1)) * PT_ROW + 8 * kq) * 2 + 64 * kb2);
            const u32x4 az = *reinterpret_cast<const u32x4*>(azp + 64 * kb2);
            accz = mfma_f16(az, pw, accz);
            const u32x4 sw = *reinterpret_cast<const u32x4*>(sm + Lds::OFF_VS + 16 * kq + 64 * kb2);
            const uint8_t* const vp = sm + Lds::OFF_VT + (j >> 3) * VT_COL * 4 + 32 * kq + 128 * kb2;
            const u32x4 va = *reinterpret_cast<const u32x4*>(vp), vbb = *reinterpret_cast<const u32x4*>(vp + 16);
            const uint32_t mg[4] = {__builtin_amdgcn_perm(va[1], va[0], vsel), __builtin_amdgcn_perm(va[3], va[2], vsel),
                                    __builtin_amdgcn_perm(vbb[1], vbb[0], vsel), __builtin_amdgcn_perm(vbb[3], vbb[2], vsel)};
            const uint32_t up = 8u - 2u * (j & 3), dn = 2u * (j & 3);
            u32x4 lo, hi;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                lo[i] = k_or(mg[i] << up, 0x03000300u, sw[i]);
                hi[i] = k_or(mg[i] >> dn, 0x03000300u, sw[i]);
            }
            acc[0] = mfma_f16(lo, pw, acc[0]);
            acc[1] = mfma_f16(hi, pw, acc[1]);
            if constexpr (FINE) {
                const u32x4 pl = *reinterpret_cast<const u32x4*>(sm + Lds::OFF_PL + ((j & (NH - 1)) * PT_ROW + 8 * kq) * 2 + 64 * kb2);
                accz = mfma_f16(az, pl, accz);
                acc[0] = mfma_f16(lo, pl, acc[0]);
                acc[1] = mfma_f16(hi, pl, acc[1]);
            }
        }
        lds_fence();
    }
    const int errors = (any_lane(bad_id) ? OMMX_ERR_TABLE_RANGE : 0) | (over_step ? OMMX_ERR_VALUE_RANGE : 0);
    if (__builtin_expect(errors, 0)) {
        int32_t* const err = args_again().err;
        if (err && lane == 0) atomicOr(err, errors);
    }

    // ---- the state: o = (4 (acc - sum p*2^e) + sum p*zp) / l, lse = m + ln l ------------------------------------------
    const float sz = lane_value(accz[0], j), ss = lane_value(accz[1], j), l_tot = lane_value(accz[2], j);
    const float inv = l_tot > 0.0f ? __builtin_amdgcn_rcpf(l_tot) : 0.0f;
    const int h = j & (NH - 1), x = NH == 8 ? j >> 3 : j >> 2;            // head and replica of the column
    if (h < R) {
        const uint32_t dst = h * al_h + 64 * (kq >> 1) + 32 * (kq & 1);
        auto val = [&](float v) { return (4.0f * (v - ss) + sz) * inv; };
        auto put = [&](uint32_t at, float v, float w) { tail::put2<true>(reinterpret_cast<float*>(al + at), val(v), val(w)); };
        if constexpr (NH == 4) {           // four replicas: two channels each
            const f32x4 mine = (x & 1) ? acc[1] : acc[0];
            put(dst + 16 * (x & 1) + 4 * (x & 2), (x & 2) ? mine[2] : mine[0], (x & 2) ? mine[3] : mine[1]);
        } else {
            const f32x4 mine = x ? acc[1] : acc[0];
            put(dst + 16 * x, mine[0], mine[1]);
            put(dst + 16 * x + 8, mine[2], mine[3]);
        }
        if (x == 0 && kq == (NH == 8 ? (h >> 2) : 0) && (HALF ? (wave & 1) : wave) == 0) {
            const int hr = h & 3;
            const float mt = hr == 0 ? m_run[0] : (hr == 1 ? m_run[1] : (hr == 2 ? m_run[2] : m_run[3]));
            tail::put1<true>(reinterpret_cast<float*>(sl + h * sl_h),
                             l_tot > 0.0f ? (mt + __builtin_amdgcn_logf(l_tot)) * 0.6931471805599453f : -INFINITY);
        }
    }
}

// ---- the merge inside the launch ------------------------------------------------------------------------------------------
// The last workgroup of a kv head to arrive merges its states: o = sum w_i o_i / sum w_i, w_i = exp(lse_i - max), as fold_kernel
// (ommx_combine.hip) does, in the order of the states whoever it is.
// States and lse are stored past the die's own cache (agent scope); a wave waits for its stores before the workgroup counts itself,
// and whoever comes last reads past its caches too.  No fences: one before the count would write a die's whole cache back (10 us), one
// after it drop what the caches hold (0.7 to 2 us).  The count lies in the call's own scratch, which nobody has cleared: a call has a number of its own, larger than nearly
// everything that memory may hold, to which every workgroup raises the word (number << 8 | arrived) when it starts.  (The number
// comes with the launch, so a launch that is replayed has no place here: under capture the merge is a launch of its own.)
// Flags of all states, looked at by everybody, need no count, but nearly all see the last one: 8 requests of 97 to 701 tokens
// 14 us instead of 10.
// How many workgroups have counted themselves before this one; `seen`: the word before this one raised it.
__device__ __forceinline__ unsigned long long arrive(unsigned long long* word, unsigned long long number, unsigned long long seen) {
    // (a word that was above this call's number is brought down to it; from then on it holds the number, whoever got it there)
    while ((seen >> 8) > number &&
           !__hip_atomic_compare_exchange_strong(word, &seen, number << 8, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
    }
    return __hip_atomic_fetch_add(word, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & 255u;
}

constexpr int MOST_STATES = kTeamMerged + kTailParts;       // of a head (a state a lane; registers and code for all of them)

// A wave takes a head (of 64 channels two at a time), LPR lanes a state, and works out the weights with a state a lane: the waves
// exchange nothing.
template <int DH>
__device__ __forceinline__ void merge_states(const TeamArgs& a, int b, int qh0, int heads, int n, int lane, int wave) {
    constexpr int LPR = DH / 4, ROWS = 64 / LPR, LOADS = MOST_STATES / ROWS, HP = DH == 64 ? 2 : 1;
    static_assert(MOST_STATES <= 64 && MOST_STATES % ROWS == 0, "a state a lane");
    const int front = a.tails ? kTailParts : 0;           // states of the tail, before the others
    const uint32_t N = min(n + front, MOST_STATES);
    const int c4 = lane % LPR, row = lane / LPR;
    // (bytes; a request's states span less than 2^32 of them)
    const uint32_t al_h = 4u * a.al_h, al_s = 4u * a.al_s, sl_h = 4u * a.sl_h, sl_s = 4u * a.sl_s;
    const char* const al = reinterpret_cast<const char*>(a.al) + b * 4u * a.al_b - front * static_cast<int64_t>(al_s);
    const char* const sl = reinterpret_cast<const char*>(a.sl) + b * 4u * a.sl_b - front * static_cast<int64_t>(sl_s);
    for (int h0 = wave; h0 < heads; h0 += WAVES * HP) {
        float lse[HP];
        uint64_t v[HP][LOADS][2];
#pragma unroll
        for (int k = 0; k < HP; ++k)
            lse[k] = __hip_atomic_load(reinterpret_cast<const float*>(sl + ((qh0 + min(h0 + WAVES * k, heads - 1)) * sl_h + min(static_cast<uint32_t>(lane), N - 1) * sl_s)),
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int k = 0; k < HP; ++k) {
            uint32_t at = (qh0 + min(h0 + WAVES * k, heads - 1)) * al_h + 16u * c4;
            const uint32_t end = at + (N - 1) * al_s;
            at += row * al_s;
#pragma unroll
            for (int i = 0; i < LOADS; ++i) {
                v[k][i][0] = v[k][i][1] = 0;
                if (static_cast<uint32_t>(i * ROWS) < N) {
                    const uint64_t* const from = reinterpret_cast<const uint64_t*>(al + min(at, end));
#pragma unroll
                    for (int w = 0; w < 2; ++w) v[k][i][w] = __hip_atomic_load(from + w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                at += ROWS * al_s;
            }
        }
#pragma unroll
        for (int k = 0; k < HP; ++k) {
            const int h = h0 + WAVES * k;
            if (h >= heads) break;
            if (lane >= static_cast<int>(N)) lse[k] = -INFINITY;
            const float tops = tail::row16_max(lse[k]);
            const float top = fmaxf(fmaxf(readlane_f32(tops, 0), readlane_f32(tops, 16)), fmaxf(readlane_f32(tops, 32), readlane_f32(tops, 48)));
            const float w = lse[k] == -INFINITY ? 0.0f : __expf(lse[k] - top);
            const float sums = tail::row16_sum(w);
            const float W = (readlane_f32(sums, 0) + readlane_f32(sums, 16)) + (readlane_f32(sums, 32) + readlane_f32(sums, 48));
            float ws[LOADS];
#pragma unroll
            for (int i = 0; i < LOADS; ++i) ws[i] = lane_value(w, i * ROWS + row);        // (zero past the last state)
            // (a state of weight zero may hold anything)
            if (__builtin_expect(__popcll(__ballot(w != 0.0f)) != static_cast<int>(N), 0)) {
#pragma unroll
                for (int i = 0; i < LOADS; ++i)
                    if (ws[i] == 0.0f) v[k][i][0] = v[k][i][1] = 0;
            }
            f32x4 acc = {0, 0, 0, 0};
#pragma unroll
            for (int i = 0; i < LOADS; ++i)
#pragma unroll
                for (int c = 0; c < 4; ++c) acc[c] = fmaf(ws[i], __uint_as_float(static_cast<uint32_t>(v[k][i][c >> 1] >> (32 * (c & 1)))), acc[c]);
            const float inv = W > 0.0f ? 1.0f / W : 0.0f;
            const float x = tail::fold32(acc[0], acc[2]) * inv, y = tail::fold32(acc[1], acc[3]) * inv;
            const int64_t to = b * a.o_b + (int64_t)(qh0 + h) * a.o_h + 4 * c4 + 2 * (lane >> 5);
            if constexpr (LPR == 32) {
                if (a.o16) {
                    a.o16[to] = f32_to_bf16_any(x);
                    a.o16[to + 1] = f32_to_bf16_any(y);
                } else {
                    a.o[to] = x;
                    a.o[to + 1] = y;
                }
            } else {
                const float z = tail::fold16(x, y);
                if (a.o16) a.o16[to + (row & 1)] = f32_to_bf16_any(z);
                else a.o[to + (row & 1)] = z;
            }
            if (lane == 0) a.lse[b * a.lse_b + qh0 + h] = W > 0.0f ? top + __logf(W) : -INFINITY;
        }
    }
}

// IDX, OWN_MAP: as in ommx_decode_gqa4.hip.  NH: q heads of a kv head the matrix rows are laid out for, 4 (1, 2 or 4 of them) or
// 8.  HALF: head_dim 64, a workgroup takes a pair of kv heads, two waves each.  DEALT: the work of several requests in equal
// shares (ommx_decode_shares.h), else a.S splits each.  The first workgroups of a kv head (HALF: two) attend its bf16 tail rows, if there are any.
template <int IDX, bool OWN_MAP, int NH, bool HALF, bool DEALT>
__global__ void __launch_bounds__(64 * WAVES, team_resident(NH)) decode_team_kernel(TeamArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int unit = DEALT ? blockIdx.x : blockIdx.y;
    const int first = DEALT ? a.tails * a.B : a.tails;
    const int at = DEALT ? blockIdx.y : blockIdx.x;
    int b, page = 0, slot = 0;
    uint32_t n;                                     // splits of the request that hold something
    // (first of all: a wait for a load waits for what was asked for before it too, and this is through before any row is)
    unsigned long long seen = 0;
    auto announce = [&]() {
        if (a.arrivals && threadIdx.x == 0)
            seen = __hip_atomic_fetch_max(a.arrivals + 8 * (b * a.Hkv + unit), a.number << 8, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    if (at < first) {
        const TeamArgs& t = args_again();
        b = DEALT ? (HALF ? at >> 1 : at) : blockIdx.z;
        announce();
        uint8_t* const sm = smem + wave * TeamLds<NH, !OWN_MAP>::LDS_WAVE;
        if constexpr (HALF) tail::attend_part<NH, 64, true>(t, sm, b, 2 * unit + (at & 1), t.heads >> 1, wave, lane);
        else tail::attend_part<NH, 128, true>(t, sm, b, unit, t.heads, wave, lane);
        if (!t.arrivals) return;
        if constexpr (DEALT) {
            shares::Share mine;
            shares::find_share<32, 1, true>(t, b, lane, mine);
            n = mine.n;
        } else {
            const uint32_t G = static_cast<uint32_t>(max(t.seq[b], 0) + 31) >> 5, S = t.S, per = max(static_cast<uint32_t>(t.per), (G + S - 1) / S);
            n = (G + per - 1) / per;
        }
    } else {
        uint32_t sp, g_first, g_count;
        int L;
        if constexpr (DEALT) {
            shares::Share mine;
            if (!shares::find_share<32, 1>(a, at - first, lane, mine)) return;
            b = mine.b; L = mine.L; sp = mine.sp; n = mine.n;
            announce();
            if (sp == 0 && !a.arrivals) {
                // the merge then goes by the lse alone: the slots this request does not use say that nothing was attended
                for (int r = wave; r < a.heads; r += WAVES)
                    for (uint32_t s = n + lane; s < static_cast<uint32_t>(a.S); s += 64)
                        a.sl[b * a.sl_b + (unit * a.heads + r) * a.sl_h + s * a.sl_s] = -INFINITY;
            }
            const uint32_t G = static_cast<uint32_t>(max(L, 0) + 31) >> 5, each = G / n, more = G - each * n;
            g_first = sp * each + min(sp, more);
            g_count = each + (sp < more ? 1u : 0u);
        } else {
            b = blockIdx.z; sp = at - first;
            announce();
            // `per` groups a split: where it starts is known before the length is, and its tables are asked for at once
            uint32_t per = a.per;
            g_first = sp * per;
            page = *reinterpret_cast<const int*>(a.rt + b * a.rt_b + ((uint32_t)min((static_cast<int>(g_first << 5) + lane + a.tok_off) >> a.ps_sh, a.rt_n - 1) << a.tsh));
            slot = *reinterpret_cast<const int*>(a.rg + b * a.rg_b + ((uint32_t)min(static_cast<int>(g_first) + (lane >> 5), a.rg_n - 1) << a.tsh));
            L = a.seq[b];
            const uint32_t G = static_cast<uint32_t>(max(L, 0) + 31) >> 5, S = a.S;
            if (G > S * per) {                      // longer than the caller said: more in every split, and other tables
                per = (G + S - 1) / S;
                g_first = sp * per;
                page = *reinterpret_cast<const int*>(a.rt + b * a.rt_b + ((uint32_t)((min(static_cast<int>(g_first << 5) + lane, max(L, 1) - 1) + a.tok_off) >> a.ps_sh) << a.tsh));
                slot = *reinterpret_cast<const int*>(a.rg + b * a.rg_b + ((uint32_t)min(g_first + (lane >> 5), G - 1) << a.tsh));
            }
            n = (G + per - 1) / per;
            if (n == 0 && a.tails == 0) n = 1;      // (somebody has to say that nothing was attended)
            g_count = g_first < G ? min(per, G - g_first) : 0u;
        }
        if (L < 0) {                                // a negative length: nothing packed, reported
            L = 0;
            report_table_range(a.err, true);
        }
        if (g_count == 0) {                         // an empty split: nothing attended (what the state holds is not read then)
            for (int r = threadIdx.x; r < a.heads; r += 64 * WAVES)
                tail::put1<true>(a.sl + b * a.sl_b + (unit * a.heads + r) * a.sl_h + sp * a.sl_s, -INFINITY);
            if (a.tails == 0 && !a.arrivals) {      // (a merge of its own without a tail multiplies it by its weight, zero)
                const int width = HALF ? D / 2 : D;
                for (int i = threadIdx.x; i < a.heads * width; i += 64 * WAVES)
                    a.al[b * a.al_b + (unit * a.heads + i / width) * a.al_h + sp * a.al_s + i % width] = 0.0f;
            }
            if (!DEALT && !(a.tails == 0 && sp == 0)) return;      // (one of a fixed number is not waited for)
        } else {
            walk<IDX, OWN_MAP, NH, HALF>(a, smem, unit, b, L, sp, g_first, g_count, page, slot, !DEALT, lane, wave);
        }
    }
    const TeamArgs& t = args_again();
    if (!t.arrivals) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    team_barrier();
    const int heads = t.heads;
    uint32_t* const s_arrived = reinterpret_cast<uint32_t*>(smem);
    if (threadIdx.x == 0) *s_arrived = static_cast<uint32_t>(arrive(t.arrivals + 8 * (b * t.Hkv + unit), t.number, seen));
    team_barrier();
    const bool last = *s_arrived == n + t.tails - 1;
    if (!last) return;
    merge_states<HALF ? 64 : 128>(t, b, unit * heads, heads, n, lane, wave);
}

}  // namespace

// Returns 0 when launched, 1 when the shape belongs to another kernel (the same bounds as launch_decode_gqa4's).
int launch_decode_team(const DecodeArgs& a, int Dh, int R, const DecodeTail* tail, const TeamMerge& merge, hipStream_t st) {
    if (a.scale_bf16 || a.v_bf16 || a.gt != 32 || a.gc != 32 || a.kout != 6) return 1;
    if ((reinterpret_cast<uintptr_t>(a.q) & 3) || (a.q_sb & 1) || (a.q_sh & 1)) return 1;
    const bool half = Dh == 64;
    if (half ? !(R == 1 || R == 2 || R == 4) || a.Hkv % 2 || a.idx_repr != 0 : Dh != 128 || !(R == 1 || R == 2 || R == 4 || R == 8)) return 1;
    const int Hk = half ? a.Hkv / 2 : a.Hkv;
    const uint64_t lim = 0xFFFFFF00ull;
    if (a.n_pages <= 0 || a.n_gslots <= 0 || static_cast<uint64_t>(a.n_pages) * static_cast<uint64_t>(a.ps) >= (1ull << 24) ||
        static_cast<uint64_t>(a.n_pages) * a.ps * Hk * 32ull > lim || static_cast<uint64_t>(a.n_gslots) * Hk * D * 6ull > lim)
        return 1;
    if (a.shares > 0 ? a.B > 64 : merge.per_split < 1) return 1;
    // 32-bit offsets behind scalar bases: no stride below zero, and everything they reach within 2^32 bytes
    const int tsh = a.i64 ? 3 : 2;
    const auto reach = [&](int64_t b, int64_t h, int64_t s, int64_t bytes) {
        return b >= 0 && h >= 0 && s >= 0 && b <= lim && h <= lim && s <= lim && (a.B * b + a.Hq * h + (a.S + kTailParts) * s + 256) * bytes <= static_cast<int64_t>(lim);
    };
    if (!reach(a.q_sb, a.q_sh, 0, 2) || a.q_sh >= (1 << 22) || !reach(a.al_b, a.al_h, a.al_s, 4) || !reach(a.sl_b, a.sl_h, a.sl_s, 4) ||
        !reach(a.rt_s, 0, 0, 8) || !reach(a.rg_s, 0, 0, 8) || merge.rt_n < 1 || merge.rg_n <= a.gbase)
        return 1;
    // (states are written and merged eight bytes at a time and more)
    if ((reinterpret_cast<uintptr_t>(a.al) & 15) || a.al_b % 4 || a.al_h % 4 || a.al_s % 4) return 1;
    if (merge.arrivals && (a.S > kTeamMerged || !merge.lse || merge.number < kFirstCall)) return 1;
    const int nh = R == 8 ? 8 : 4, tails = !tail ? 0 : half ? 2 : 1;
    auto u = [](int64_t v) { return static_cast<uint32_t>(v); };
    const TeamArgs t{merge.arrivals, merge.number, merge.o, merge.o16, merge.lse, merge.o_b, merge.o_h, merge.lse_b,
                     a.seq, a.q, a.k_base, a.k_scale, a.k_zp, a.k_ms, a.k_mc, a.k_obmp, a.k_oval, a.v_main, a.v_scale, a.v_zp,
                     static_cast<const char*>(a.rt), static_cast<const char*>(a.rg) + (static_cast<int64_t>(a.gbase) << tsh), a.al, a.sl, a.err,
                     u(a.rt_s << tsh), u(a.rg_s << tsh), merge.rt_n, merge.rg_n - a.gbase,
                     u(a.q_sb), u(a.q_sh), u(a.al_b), u(a.al_h), u(a.al_s), u(a.sl_b), u(a.sl_h), u(a.sl_s),
                     a.Hq / Hk, Hk, __builtin_ctz(a.ps), tsh, a.gbase * 32 + a.off, a.n_pages, a.n_gslots, a.S, merge.per_split,
                     a.sm_scale, a.cap, a.B, a.shares, a.shares_few, a.singles, a.share_count, tails, tail ? *tail : DecodeTail{}};
    const dim3 grid = a.shares > 0 ? dim3(Hk, a.shares + tails * a.B) : dim3(a.S + tails, Hk, a.B);
    const size_t shm = nh == 8 ? (a.k_ms ? TeamLds<8, false>::BYTES : TeamLds<8, true>::BYTES) : a.k_ms ? TeamLds<4, false>::BYTES : TeamLds<4, true>::BYTES;
#define OMMX_TEAM(IDX, MAP, NH, HALF)                                                                                            \
    do {                                                                                                                         \
        if (a.shares > 0) hipLaunchKernelGGL((decode_team_kernel<IDX, MAP, NH, HALF, true>), grid, dim3(64 * WAVES), shm, st, t);  \
        else hipLaunchKernelGGL((decode_team_kernel<IDX, MAP, NH, HALF, false>), grid, dim3(64 * WAVES), shm, st, t);              \
    } while (0)
    const int form = (half ? 8 : 0) | (nh == 8 ? 4 : 0) | (a.idx_repr ? 2 : 0) | (a.k_ms ? 1 : 0);
    switch (form) {
        case 0: OMMX_TEAM(0, false, 4, false); break;
        case 1: OMMX_TEAM(0, true, 4, false); break;
        case 2: OMMX_TEAM(1, false, 4, false); break;
        case 3: OMMX_TEAM(1, true, 4, false); break;
        case 4: OMMX_TEAM(0, false, 8, false); break;
        case 5: OMMX_TEAM(0, true, 8, false); break;
        case 6: OMMX_TEAM(1, false, 8, false); break;
        case 7: OMMX_TEAM(1, true, 8, false); break;
        case 8: OMMX_TEAM(0, false, 4, true); break;
        default: OMMX_TEAM(0, true, 4, true); break;
    }
#undef OMMX_TEAM
    return 0;
}

}  // namespace ommx
