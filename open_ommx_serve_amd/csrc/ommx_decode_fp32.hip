// Split-KV decode kernel in fp32 for 64-channel heads with position streams (32 / 64 / 128-token groups, up to ten outliers, 1, 2
// or 4 q heads per kv head, int8 exponents, INT2 V).  Same operator and arithmetic as the plain kernel (ommx_decode_ref.hip,
// reference ommx_gpu_serve/attention/paged_decode.py:1657-2284), which served these calls before: K and V dequantised to fp32,
// fp32 products and sums, no 16-bit operand anywhere.
//
// What bounded that one: a workgroup per kv head and 32 tokens with six barriers a tile, four loads in a chain, a byte of V
// and two parameters per four products.  Here a wave owns one kv head of one split and walks it 64 tokens a step without
// meeting another, the next step's rows and parameters on their way meanwhile, and the products run on
// v_mfma_f32_4x4x1, whose operands are what the lanes have anyway:
//   * logits: lane = token.  Sixteen blocks of four tokens, B the token's own K value, A channel c of the four q heads
//     (lane & 3 is the head); the result is the lane's own token for all heads.  K passes through LDS as an fp32 tile of 32 channels, where
//     the outliers (lane = channel) replace the base values (lane = token), as the plain kernel has it;
//   * P.V: lane = channel.  B is the channel's V value of one token, A that token's weights of the four heads; the result is the
//     lane's own channel for all heads: four sums a step that start at zero, then one addition to the running sum.
// Sums are shorter than the plain kernel's (chains of 16, and one addition per 64 tokens instead of one per sixteen): its error
// against 64 bits times 0.91 / 0.98 / 0.94 for outputs and 1.0 / 0.91 / 0.87 for the lse (32 x 32, 64 x 64 and 128-token vectors, 18 batches).
//
// Bound by what a wave issues, some 750 vector and 128 matrix instructions and 170 LDS accesses a step, at three waves a SIMD (11 KB of
// LDS a wave).  Whole call with 32 q and 8 kv heads, plain kernel -> this, 32-token streams / 64 x 64 / 128 tokens and ten outliers, us:
//   1 K tokens       14.7 -> 10.0    19.5 -> 9.8     33.6 -> 10.6
//   2 x 12 K         63.5 -> 20.3    59.8 -> 17.4    72.5 -> 18.8
//   16 of 2 to 16 K  471 -> 55.4     450 -> 49.1     482 -> 56.2
//   64 K             154 -> 31.0     146 -> 28.4     160 -> 31.9
#include "ommx_decode_shares.h"
#include "ommx_decode_tail.h"
#include "ommx_decode_util.h"

namespace ommx {

namespace {

using namespace decode_util;

constexpr int D = 64, NH = 4;
constexpr int TILE_ROW = 36;             // floats of a tile row (32 used): rows read and written as b128 by neighbouring lanes
constexpr int SPARE_ROW = 64;            // behind the 64 tokens: for outliers of other pieces of the group, and of empty slots
constexpr int HEAD_ROW = 68;             // floats of a row of [q head][64 channels or tokens]
constexpr int VT_ROW = 80;               // bytes of a V code column (64 tokens)
// LDS of a wave.  What P.V needs lies where the K tile was.
constexpr int OFF_Q = 0;                                        // [NH][HEAD_ROW] f32
constexpr int OFF_PAR = OFF_Q + NH * HEAD_ROW * 4;              // [2 halves of the step][steps, zero points][32 channels] f32
constexpr int OFF_TILE = OFF_PAR + 512;                         // [64 tokens + 1][TILE_ROW] f32
constexpr int OFF_P = OFF_TILE;                                 // [NH][HEAD_ROW] f32 softmax weights
constexpr int OFF_VP = OFF_P + NH * HEAD_ROW * 4;               // [2 V vectors][64 tokens]{step, zero point}
constexpr int OFF_VT = OFF_VP + 1024;                           // [16 code bytes of a row][VT_ROW]
constexpr int LDS_WAVE = OFF_TILE + 65 * TILE_ROW * 4;          // 10960
static_assert(OFF_PAR % 16 == 0 && OFF_TILE % 16 == 0 && OFF_VP % 16 == 0 && OFF_VT % 16 == 0 && LDS_WAVE % 16 == 0, "b128 alignment");
static_assert(OFF_VT + 16 * VT_ROW <= LDS_WAVE && (32 * NH + 2 * NH) * 4 <= LDS_WAVE, "P.V and the tail rows fit");
constexpr int RESIDENT = 3;              // workgroups a compute unit, by LDS (in pieces of 1280 bytes) and registers
static_assert(RESIDENT * ((4 * LDS_WAVE + 1279) / 1280 * 1280) <= 160 * 1024, "LDS");

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 0, 0, 0); }
// Bits [at, at + 7) of the position stream
template <int N>
__device__ __forceinline__ uint32_t field7(const uint32_t (&x)[N], int at) {
    const int w = at >> 5, s = at & 31;
    return (s > 25 && w + 1 < N ? __builtin_amdgcn_alignbit(x[w + 1], x[w], s) : x[w] >> s) & 127u;
}

// SLOTS: outlier slots walked, 6 or 10 (a.kout of them used).  GTS: groups of 32 << GTS tokens; longer ones are dealt out and walked
// in pieces of 64 tokens, the slots of a channel shared between the two lanes that have it.  DEALT: equal shares
// (ommx_decode_shares.h), else a.S splits of every request.
template <int SLOTS, int GTS, bool OWN_MAP, bool DEALT>
__global__ void __launch_bounds__(256, RESIDENT) decode_fp32_kernel(DecodeArgs a) {
    constexpr bool LONG = GTS > 0;
    constexpr int GT_SH = 5 + GTS, UNIT_SH = LONG ? 6 : 5;
    constexpr int NIX = SLOTS == 6 ? 2 : 3;             // dwords that hold a channel's positions, wherever they start
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    uint8_t* const sm = smem + wave * LDS_WAVE;
    const int Hkv = a.Hkv, R = a.Hq / Hkv, kvh = (DEALT ? blockIdx.x : blockIdx.y) * waves + wave, qh0 = kvh * R;
    {
        // the last workgroups of the grid attend the bf16 tail rows
        const int past = DEALT ? static_cast<int>(blockIdx.y) - a.shares : static_cast<int>(blockIdx.z) - a.B;
        if (past >= 0) {
            const int at = DEALT ? past : past * a.S + static_cast<int>(blockIdx.x);
            if (at < a.t_slices) tail::attend_part<NH, D>(a, sm, at / kTailParts, kvh, R, at & (kTailParts - 1), lane);
            return;
        }
    }
    uint32_t sp = blockIdx.x, S = static_cast<uint32_t>(a.S);
    int b = blockIdx.z, L;
    if constexpr (DEALT) {
        shares::Share mine;
        if (!shares::find_share<(1 << UNIT_SH), 1>(a, blockIdx.y, lane, mine)) return;
        b = mine.b; L = mine.L; sp = mine.sp; S = mine.n;
        if (a.t_slices && sp == 0) {
            // the merge then goes by the lse alone: the slots this request does not use say that nothing was attended
            for (int r = 0; r < R; ++r)
                for (uint32_t s = S + lane; s < static_cast<uint32_t>(a.S); s += 64)
                    a.sl[b * a.sl_b + (int64_t)(qh0 + r) * a.sl_h + (int64_t)s * a.sl_s] = -INFINITY;
        }
    } else {
        L = a.seq[b];
    }
    if (L < 0) { L = 0; report_table_range(a.err, true); }      // a negative length: nothing packed, reported
    // groups (pieces) dealt out evenly, as in ommx_decode_gqa4.hip
    const uint32_t G = static_cast<uint32_t>(L + (1 << UNIT_SH) - 1) >> UNIT_SH, each = G / S, extra = G - each * S;
    const uint32_t first = sp * each + min(sp, extra), count = each + (sp < extra ? 1u : 0u);
    const int n_begin = static_cast<int>(first << UNIT_SH), n_end = min(static_cast<int>((first + count) << UNIT_SH), L);
    float* const al = a.al + b * a.al_b + (int64_t)qh0 * a.al_h + (int64_t)sp * a.al_s;
    float* const sl = a.sl + b * a.sl_b + (int64_t)qh0 * a.sl_h + (int64_t)sp * a.sl_s;
    if (n_begin >= n_end) {                             // an empty split: the state of nothing attended
        for (int r = 0; r < R; ++r) {
            al[r * a.al_h + lane] = 0.0f;
            if (lane == 0) sl[r * a.sl_h] = -INFINITY;
        }
        return;
    }

    // ---- addressing: scalar plane pointers and 32-bit byte offsets, as in ommx_decode_gqa4.hip ------------------
    const uint32_t Hk = static_cast<uint32_t>(Hkv), row_bytes = Hk * 16u;
    const int last = n_end - 1, ps_sh = __ffs(a.ps) - 1, ps_mask = a.ps - 1, tsh = a.i64 ? 3 : 2;
    const int tok_off = (a.gbase << GT_SH) + a.off;
    const char* const rt_b = static_cast<const char*>(a.rt) + ((b * a.rt_s) << tsh);
    const char* const rg_b = static_cast<const char*>(a.rg) + ((b * a.rg_s + a.gbase) << tsh);
    const bool two_vecs = a.gc == 32;                   // V vectors of a token: two of 32 channels or one of 64
    const uint8_t* const kb = a.k_base + kvh * 16;
    const uint8_t* const vb = a.v_main + kvh * 16;
    const int8_t* const vs = a.v_scale + (two_vecs ? 2 * kvh : kvh);
    const uint16_t* const vz = a.v_zp + (two_vecs ? 2 * kvh : kvh);
    auto at = [](const void* base, uint32_t byte_off) { return static_cast<const char*>(base) + byte_off; };
    const int g = lane >> 5, c = lane & 31;             // half of the step; channel of the chunk
    const int kout = a.kout;
    const uint32_t n_ix = relidx7_bytes(kout), n_ov = static_cast<uint32_t>(kout + 1) >> 1;
    bool bad_id = false;
    int page, slot;
    auto fetch_tables = [&](int n) {
        page = *reinterpret_cast<const int*>(rt_b + ((uint32_t)((min(n + lane, last) + tok_off) >> ps_sh) << tsh));
        slot = *reinterpret_cast<const int*>(rg_b + ((uint32_t)(LONG ? min(n, last) >> GT_SH : min((n >> 5) + g, last >> 5)) << tsh));
    };
    u32x4 kr, vr;
    uint32_t row = 0, vsc, vzp;
    auto fetch_k = [&](int n) {
        page = clamp_id(page, a.n_pages, bad_id);
        row = __umul24(static_cast<uint32_t>((page << ps_sh) + ((min(n + lane, last) + tok_off) & ps_mask)), row_bytes);
        kr = *reinterpret_cast<const u32x4*>(at(kb, row));
    };
    auto fetch_v = [&]() {
        vr = *reinterpret_cast<const u32x4*>(at(vb, row));
        if (two_vecs) {
            vsc = *reinterpret_cast<const uint16_t*>(at(vs, row >> 3));
            vzp = *reinterpret_cast<const uint32_t*>(at(vz, row >> 2));
        } else {
            vsc = *reinterpret_cast<const uint8_t*>(at(vs, row >> 4));
            vzp = *reinterpret_cast<const uint16_t*>(at(vz, row >> 3));
        }
    };
    // parameters of channel c of either chunk, for the lane's half of the step
    uint32_t p_sc[2], p_zp[2], p_ms[2], p_mc[2], p_ix[2][NIX], p_ov[2][2], p_ch;
    auto fetch_params = [&]() {
        p_ch = (static_cast<uint32_t>(clamp_id(slot, a.n_gslots, bad_id)) * Hk + kvh) * D + c;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint32_t ch = p_ch + 32 * u;
            p_sc[u] = *reinterpret_cast<const uint8_t*>(at(a.k_scale, ch));
            p_zp[u] = *reinterpret_cast<const uint16_t*>(at(a.k_zp, 2 * ch));
            if (OWN_MAP) {
                p_ms[u] = *reinterpret_cast<const uint16_t*>(at(a.k_ms, 2 * ch));
                p_mc[u] = *reinterpret_cast<const uint16_t*>(at(a.k_mc, 2 * ch));
            }
            // (the aligned dwords that hold the channel's bytes, and no others)
            const uint32_t ix = ch * n_ix, ov = ch * n_ov, ix_last = (ix + n_ix - 1) & ~3u, ov_last = (ov + n_ov - 1) & ~3u;
#pragma unroll
            for (int i = 0; i < NIX; ++i) p_ix[u][i] = *reinterpret_cast<const uint32_t*>(at(a.k_obmp, min((ix & ~3u) + 4 * i, ix_last)));
#pragma unroll
            for (int i = 0; i < 2; ++i) p_ov[u][i] = *reinterpret_cast<const uint32_t*>(at(a.k_oval, min((ov & ~3u) + 4 * i, ov_last)));
        }
    };
    fetch_tables(n_begin);
    asm volatile("" ::: "memory");
    float* const s_q = reinterpret_cast<float*>(sm + OFF_Q);
#pragma unroll
    for (int h = 0; h < NH; ++h)
        s_q[h * HEAD_ROW + lane] = bf16_to_f32(a.q[b * a.q_sb + (int64_t)(qh0 + min(h, R - 1)) * a.q_sh + lane]);
    fetch_k(n_begin);
    fetch_params();
    fetch_v();
    if (n_begin + 64 < n_end) fetch_tables(n_begin + 64);
    asm volatile("" ::: "memory");

    float* const s_par = reinterpret_cast<float*>(sm + OFF_PAR);
    float* const s_tile = reinterpret_cast<float*>(sm + OFF_TILE);
    f32x4 acc = {0, 0, 0, 0};
    float m_run[NH], l_run[NH];                         // l_run: of the lane's tokens
#pragma unroll
    for (int h = 0; h < NH; ++h) { m_run[h] = -INFINITY; l_run[h] = 0.0f; }
    const uint32_t not_first = lane >= 32 ? 128u : 0u;

    for (int n0 = n_begin; n0 < n_end; n0 += 64) {
        const bool more = n0 + 64 < n_end, second = n0 + 32 < n_end;
        // ------------------------------------------------------------------ logits, 32 channels at a time
        f32x4 d[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) d[i] = f32x4{0, 0, 0, 0};
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const float step = __uint_as_float(static_cast<uint32_t>(static_cast<int8_t>(p_sc[u]) + 127) << 23);
            const float zp = __uint_as_float(p_zp[u] << 16);
            s_par[64 * g + c] = step;
            s_par[64 * g + 32 + c] = zp;
            lds_fence();
            {   // base values, lane = token
                f32x4* const to = reinterpret_cast<f32x4*>(s_tile + lane * TILE_ROW);
                const f32x4* const ps = reinterpret_cast<const f32x4*>(s_par + 64 * g);
#pragma unroll
                for (int w = 0; w < 2; ++w) {
                    uint32_t m[4];                      // byte i of m[j]: the code of channel 16 w + 4 i + j
#pragma unroll
                    for (int s = 0; s < 4; ++s) m[s] = (kr[2 * u + w] >> (2 * s)) & 0x03030303u;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const f32x4 st = ps[4 * w + i], z = ps[8 + 4 * w + i];
                        f32x4 k;
#pragma unroll
                        for (int s = 0; s < 4; ++s) k[s] = fmaf(static_cast<float>((m[s] >> (8 * i)) & 0xFFu), st[s], z[s]);
                        to[4 * w + i] = k;
                    }
                }
            }
            lds_fence();
            {   // outliers, lane = channel of either half
                uint32_t x[NIX], y[2];
                const uint32_t ch = p_ch + 32 * u, xs = 8 * ((ch * n_ix) & 3) + (LONG ? 7 * g : 0), ys = 8 * ((ch * n_ov) & 3) + (LONG ? 4 * g : 0);
#pragma unroll
                for (int i = 0; i < NIX; ++i) x[i] = i + 1 < NIX ? __builtin_amdgcn_alignbit(p_ix[u][i + 1], p_ix[u][i], xs) : p_ix[u][i] >> xs;
                y[0] = __builtin_amdgcn_alignbit(p_ov[u][1], p_ov[u][0], ys);
                y[1] = p_ov[u][1] >> ys;
                // level / map_scale: the quotient of 1 or 1.5, correctly rounded, times a power of two
                float r1 = 0, r3 = 0, mc = 0;
                if (OWN_MAP) {
                    const float ms = __uint_as_float(p_ms[u] << 16);
                    r1 = __fdiv_rn(1.0f, ms);
                    r3 = __fdiv_rn(1.5f, ms);
                    mc = __uint_as_float(p_mc[u] << 16);
                }
                auto put = [&](uint32_t to, float level) {
                    float k;
                    if (OWN_MAP) {
                        const uint32_t bits = __float_as_uint(level);
                        k = fmaf(__uint_as_float(bits & 0xFF800000u), (bits & 0x00400000u) ? r3 : r1, mc);
                    } else {
                        k = fmaf(level, step, zp);
                    }
                    s_tile[to * TILE_ROW + c] = k;
                };
                // (position streams hold values up to 127: one outside the tile, and a slot beyond kout, goes to the spare row)
                if constexpr (!LONG) {
#pragma unroll
                    for (int s = 0; s < SLOTS; ++s) {
                        const uint32_t pos = field7(x, 7 * s);
                        const uint32_t byte = y[s >> 3] >> (8 * ((s >> 1) & 3));
                        const f32x2 lv = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(byte, 1.0f, 0);
                        put(s < kout && pos < 32u ? 32u * g + pos : static_cast<uint32_t>(SPARE_ROW), lv[s & 1]);
                    }
                } else {
                    const uint32_t from = GTS == 2 ? static_cast<uint32_t>(n0) & 64u : 0u;
#pragma unroll
                    for (int s = 0; s < SLOTS / 2; ++s) {           // slots 2 s + g
                        const uint32_t pos = field7(x, 14 * s);
                        uint32_t to = min(pos - from, static_cast<uint32_t>(SPARE_ROW));
                        // (a position named twice holds the later slot's value)
                        const uint32_t next = field7(x, 14 * s + 7) | not_first;
                        if (2 * s + g >= kout || (pos == next && 2 * s + 1 < kout)) to = SPARE_ROW;
                        const f32x2 lv = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(y[s >> 2] >> (8 * (s & 3)), 1.0f, 0);
                        put(to, lv[0]);
                    }
                }
            }
            if (u == 1 && more) { fetch_k(n0 + 64); fetch_params(); }
            lds_fence();
            {
                const f32x4* const kv = reinterpret_cast<const f32x4*>(s_tile + lane * TILE_ROW);
                const f32x4* const qv = reinterpret_cast<const f32x4*>(s_q + (lane & 3) * HEAD_ROW + 32 * u);
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const f32x4 k = kv[i], q = qv[i];
#pragma unroll
                    for (int s = 0; s < 4; ++s) d[2 * u + (s & 1)] = mfma_f32(q[s], k[s], d[2 * u + (s & 1)]);
                }
            }
            lds_fence();
        }
        // ------------------------------------------------------------------ softmax: lane = token, a register a head
        float x[NH];
        {
            const f32x4 sum = (d[0] + d[1]) + (d[2] + d[3]);
#pragma unroll
            for (int h = 0; h < NH; ++h) x[h] = n0 + lane < n_end ? apply_cap(sum[h] * a.sm_scale, a.cap) : -INFINITY;
        }
        float over = -INFINITY;
#pragma unroll
        for (int h = 0; h < NH; ++h) over = fmaxf(over, x[h] - m_run[h]);
        if (any_lane(over > 8.0f)) {        // (the weights are fp32: any maximum that keeps them in range serves)
            float mx[NH];
#pragma unroll
            for (int h = 0; h < NH; ++h) mx[h] = x[h];
            wave_max4(mx);
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                const float m_new = fmaxf(m_run[h], mx[h]);
                const float alpha = m_run[h] == -INFINITY ? 0.0f : __expf(m_run[h] - m_new);
                m_run[h] = m_new;
                l_run[h] *= alpha;
                acc[h] *= alpha;
            }
        }
        // ------------------------------------------------------------------ P.V
        {
            float* const s_p = reinterpret_cast<float*>(sm + OFF_P);
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                const float p = x[h] == -INFINITY ? 0.0f : __expf(x[h] - m_run[h]);
                l_run[h] += p;
                s_p[h * HEAD_ROW + lane] = p;
            }
            uint8_t* const vt = sm + OFF_VT + lane;
#pragma unroll
            for (int i = 0; i < 16; ++i) vt[i * VT_ROW] = static_cast<uint8_t>(vr[i >> 2] >> (8 * (i & 3)));
            f32x2* const vp = reinterpret_cast<f32x2*>(sm + OFF_VP) + lane;
            // (a token past the split: its V is zero, as its weight is)
            const bool live = n0 + lane < n_end;
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                const float st = __uint_as_float(static_cast<uint32_t>(static_cast<int8_t>(vsc >> (8 * v)) + 127) << 23);
                const float z = __uint_as_float(v ? vzp & 0xFFFF0000u : vzp << 16);
                if (v == 0 || two_vecs) vp[64 * v] = live ? f32x2{st, z} : f32x2{0.0f, 0.0f};
            }
        }
        if (more) {
            fetch_v();
            fetch_tables(n0 + 128);
        }
        lds_fence();
        f32x4 t[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) t[i] = f32x4{0, 0, 0, 0};
        {
            const u32x4* const codes = reinterpret_cast<const u32x4*>(sm + OFF_VT + (lane >> 2) * VT_ROW);
            const f32x4* const par = reinterpret_cast<const f32x4*>(sm + OFF_VP + (two_vecs ? 512 * g : 0));
            const f32x4* const pv = reinterpret_cast<const f32x4*>(sm + OFF_P) + (lane & 3) * (HEAD_ROW / 4);
            const uint32_t sh = 2 * (lane & 3);
#pragma unroll
            for (int blk = 0; blk < 4; ++blk) {         // 16 tokens
                if (blk == 2 && !second) break;
                const u32x4 cw = codes[blk];
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const uint32_t m = (cw[w] >> sh) & 0x03030303u;
                    const f32x4 lo = par[8 * blk + 2 * w], hi = par[8 * blk + 2 * w + 1], p = pv[4 * blk + w];
                    const float v0 = fmaf(static_cast<float>(m & 0xFFu), lo[0], lo[1]), v1 = fmaf(static_cast<float>((m >> 8) & 0xFFu), lo[2], lo[3]);
                    const float v2 = fmaf(static_cast<float>((m >> 16) & 0xFFu), hi[0], hi[1]), v3 = fmaf(static_cast<float>(m >> 24), hi[2], hi[3]);
                    t[0] = mfma_f32(p[0], v0, t[0]);
                    t[1] = mfma_f32(p[1], v1, t[1]);
                    t[2] = mfma_f32(p[2], v2, t[2]);
                    t[3] = mfma_f32(p[3], v3, t[3]);
                }
            }
        }
        acc += (t[0] + t[1]) + (t[2] + t[3]);
        lds_fence();
    }
    report_table_range(a.err, bad_id);
    wave_sum4(l_run);
#pragma unroll
    for (int h = 0; h < NH; ++h) {
        if (h >= R) break;
        const float l = l_run[h];
        al[h * a.al_h + lane] = l > 0.0f ? acc[h] / l : 0.0f;
        if (lane == 0) sl[h * a.sl_h] = l > 0.0f ? m_run[h] + __logf(l) : -INFINITY;
    }
}

template <int SLOTS, int GTS>
void launch(const DecodeArgs& a, dim3 grid, dim3 block, size_t shm, hipStream_t st) {
    switch ((a.k_ms ? 2 : 0) | (a.shares > 0 ? 1 : 0)) {
        case 0: hipLaunchKernelGGL((decode_fp32_kernel<SLOTS, GTS, false, false>), grid, block, shm, st, a); break;
        case 1: hipLaunchKernelGGL((decode_fp32_kernel<SLOTS, GTS, false, true>), grid, block, shm, st, a); break;
        case 2: hipLaunchKernelGGL((decode_fp32_kernel<SLOTS, GTS, true, false>), grid, block, shm, st, a); break;
        default: hipLaunchKernelGGL((decode_fp32_kernel<SLOTS, GTS, true, true>), grid, block, shm, st, a); break;
    }
}

}  // namespace

// Returns 0 when launched, 1 when the shape belongs to another kernel.
int launch_decode_fp32(const DecodeArgs& a_in, int Dh, int R, const DecodeTail* tail, hipStream_t st) {
    DecodeArgs a = a_in;
    if (Dh != D || !(R == 1 || R == 2 || R == 4) || a.scale_bf16 || a.v_bf16 || a.idx_repr != 1 || a.kout < 1 || a.kout > 10 ||
        !(a.gt == 32 || a.gt == 64 || a.gt == 128) || !(a.gc == 32 || a.gc == 64) || (a.gt == 32 && a.kout > 6) || a.ps > a.gt)
        return 1;
    if (a.shares > 0 && a.B > 64) return 1;
    // 32-bit byte offsets into planes whose extents are given, and whole words of them
    const uint64_t lim = 0xFFFFFF00ull;
    if (a.n_pages <= 0 || a.n_gslots <= 0 || static_cast<uint64_t>(a.n_pages) * static_cast<uint64_t>(a.ps) >= (1ull << 24) ||
        static_cast<uint64_t>(a.n_pages) * a.ps * a.Hkv * 16ull > lim || static_cast<uint64_t>(a.n_gslots) * a.Hkv * D * 9ull > lim || a.Hkv >= (1 << 20))
        return 1;
    const auto aligned = [](const void* p, uintptr_t n) { return reinterpret_cast<uintptr_t>(p) % n == 0; };
    if (!aligned(a.k_base, 16) || !aligned(a.v_main, 16) || !aligned(a.v_scale, 2) || !aligned(a.v_zp, 4) || !aligned(a.k_obmp, 4) || !aligned(a.k_oval, 4))
        return 1;
    a.t_slices = 0;
    if (tail) {
        a.t = *tail;
        a.t_slices = kTailParts * a.B;
    }
    const int waves = a.Hkv % 4 == 0 ? 4 : a.Hkv % 2 == 0 ? 2 : 1;
    const dim3 grid = a.shares > 0 ? dim3(a.Hkv / waves, a.shares + a.t_slices) : dim3(a.S, a.Hkv / waves, a.B + (a.t_slices + a.S - 1) / a.S);
    const dim3 block(64 * waves);
    const size_t shm = static_cast<size_t>(waves) * LDS_WAVE;
    if (a.gt == 32) launch<6, 0>(a, grid, block, shm, st);
    else if (a.gt == 64) { if (a.kout <= 6) launch<6, 1>(a, grid, block, shm, st); else launch<10, 1>(a, grid, block, shm, st); }
    else if (a.kout <= 6) launch<6, 2>(a, grid, block, shm, st);
    else launch<10, 2>(a, grid, block, shm, st);
    return 0;
}

}  // namespace ommx
