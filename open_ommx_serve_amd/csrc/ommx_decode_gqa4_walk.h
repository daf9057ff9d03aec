// The walk of one wave over its split, the text of two functions in ommx_decode_gqa4.hip (see there): the kernel itself, whose ANY
// is false, and other_form(), whose ANY is true.  (As a function that both call it costs the kernels of three waves a SIMD up
// to 21 spilled registers: a body that is inlined is optimised once before, without its kernel's arguments.)
    static_assert(NH == 4 || (NH == 8 && !PARTIAL), "4 heads (or fewer, PARTIAL) or exactly 8");
    static_assert(!GEN || IDX == 0, "the general form reads bitmaps");
    // outlier slots walked per vector: the general form walks 4 or 8 whatever a.kout is (loads and
    // arithmetic of all slots go out together; only the writes of the slots beyond a.kout are skipped)
    constexpr int KMAX = KSLOTS;
    static_assert(GEN ? KMAX == 4 || KMAX == 6 || KMAX == 8 : KMAX == 6 || (KMAX == 10 && GTS == 2), "outlier slots");
    static_assert(GTS == 0 || (IDX == 1 && !GEN && !PARTIAL), "longer groups are read through position streams");
    constexpr bool LONG = GTS > 0;
    constexpr int GT_SH = 5 + GTS;                    // log2 of the tokens per K group
    constexpr int UNIT_SH = LONG ? 6 : 5;             // log2 of the tokens that the work is dealt out in
    constexpr int NG = LONG ? 1 : 2;                  // groups (parameter sets) a step reads
    const int kout = GEN ? a.kout : KMAX;
    const bool half = GEN ? a.half != 0 : HALF;
    using Lds = LdsMap<NH, LONG>;
    constexpr int OFF_TILE = Lds::OFF_TILE, OFF_KT = Lds::OFF_KT, OFF_MAG = Lds::OFF_MAG, OFF_ZPP = Lds::OFF_ZPP, OFF_VT = Lds::OFF_VT,
                  OFF_PT = Lds::OFF_PT, OFF_VZ = Lds::OFF_VZ, OFF_VS = Lds::OFF_VS, OFF_LC = Lds::OFF_LC, OFF_ZERO = Lds::OFF_ZERO,
                  OFF_ONES = Lds::OFF_ONES, LDS_WAVE = Lds::LDS_WAVE;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem_all[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);     // uniform: keeps the plane pointers scalar
    uint8_t* const sm = smem_all + wave * LDS_WAVE;
    const uint32_t sm_lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
        (__attribute__((address_space(3))) uint8_t*)sm));
    const int j = lane & 15, kq = lane >> 4;
    const int Hkv = a.Hkv;
    const int waves = blockDim.x >> 6;
    // (shares: the head groups vary fastest, so that the shares nobody needs are dispatched last)
    const bool dealt = ORDER >= 1 && a.shares > 0;
    const int kvh = (dealt ? blockIdx.x : blockIdx.y) * waves + wave;
    const int heads = PARTIAL ? a.Hq / Hkv : NH;
    const int qh0 = kvh * heads;
    const int r_half = max(heads >> 1, 1);            // head_dim 64: q heads per kv head of the pair
    if (TAIL) {
        // the last workgroups of the grid attend the bf16 tail rows (head_dim 64: of either kv head of the pair)
        const int past = dealt ? static_cast<int>(blockIdx.y) - a.shares : static_cast<int>(blockIdx.z) - a.B;
        if (past >= 0) {
            const int at = dealt ? past : past * a.S + static_cast<int>(blockIdx.x);
            if (at >= a.t_slices) return;
            const int part = at & (kTailParts - 1), rest = at / kTailParts;
            const int tb = half ? rest >> 1 : rest, sub = half ? rest & 1 : 0;
            if ((GEN || HALF) && half) tail::attend_part<NH, 64>(a, sm, tb, 2 * kvh + sub, heads >> 1, part, lane);
            else if (!HALF) tail::attend_part<NH, 128>(a, sm, tb, kvh, heads, part, lane);
            return;
        }
    }
    uint32_t sp = blockIdx.x, S = static_cast<uint32_t>(a.S);
    int b = ORDER == 0 ? 0 : static_cast<int>(blockIdx.z), L;      // ORDER 0 is launched for one request only
    if (dealt) {
        shares::Share mine;
        if (!shares::find_share<(1 << UNIT_SH), ORDER == 2 ? 4 : 1>(a, blockIdx.y, lane, mine)) return;
        b = mine.b; L = mine.L; sp = mine.sp; S = mine.n;
        if (TAIL && sp == 0) {
            // the merge then goes by the lse alone: the slots this request does not use say that nothing was attended
            for (int r = 0; r < heads; ++r)
                for (uint32_t s = S + lane; s < static_cast<uint32_t>(a.S); s += 64)
                    a.sl[b * a.sl_b + (int64_t)(qh0 + r) * a.sl_h + (int64_t)s * a.sl_s] = -INFINITY;
        }
    } else if (ORDER >= 1 && a.B > 1 && a.B <= 64) {
        const int my_len = lane < a.B ? a.seq[lane] : 0;
        const uint32_t key = (static_cast<uint32_t>(my_len) << 6) | (63u - lane);
        int rank = 0;
        for (int i = 0; i < a.B; ++i)
            rank += static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(key), i)) > key;
        b = __builtin_ctzll(__ballot(lane < a.B && rank == static_cast<int>(blockIdx.z)));
        L = __builtin_amdgcn_readlane(my_len, b);
    } else if (ORDER == 2 && a.B > 1 && a.B <= 256) {
        uint32_t key[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int idx = 64 * r + lane;
            key[r] = idx < a.B ? (static_cast<uint32_t>(a.seq[idx] + 1) << 8) | (255u - idx) : 0u;
        }
        uint32_t want = 0;
        for (int bit = 31; bit >= 0; --bit) {
            const uint32_t cand = want | (1u << bit);
            int reach = 0;
#pragma unroll
            for (int r = 0; r < 4; ++r) reach += __popcll(__ballot(key[r] >= cand));
            if (reach > static_cast<int>(blockIdx.z)) want = cand;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint64_t hit = __ballot(key[r] == want);
            if (hit) b = 64 * r + __builtin_ctzll(hit);
        }
        L = static_cast<int>(want >> 8) - 1;
    } else {
        L = a.seq[b];
    }
    // q: this lane's 32 channels of head j % NH (16 dwords, channel 2i in the low half of dword i)
    // and channels 2*lane, 2*lane+1 of every head (for the channel pass)
    uint32_t qw[16], qraw[NH];      // qraw: channels 2*lane, 2*lane+1 of every head, for the thresholds below
    {
        const int hs = min(j & (NH - 1), heads - 1);
        // head_dim 64: the head's 64 channels are the pair's channels 64 * (hs / r_half) .. + 63
        const bool q_real = !half || (kq >> 1) == hs / r_half;
        const uint32_t* qh = reinterpret_cast<const uint32_t*>(
            a.q + b * a.q_sb + (int64_t)(qh0 + hs) * a.q_sh + (half ? 32 * (kq & 1) : 32 * kq));
#pragma unroll
        for (int i = 0; i < 16; ++i) qw[i] = q_real ? qh[i] : 0u;
#pragma unroll
        for (int r = 0; r < NH; ++r) {
            const int sl = min(r, heads - 1);
            const uint32_t w = *reinterpret_cast<const uint32_t*>(
                a.q + b * a.q_sb + (int64_t)(qh0 + sl) * a.q_sh + (half ? (2 * lane) & 63 : 2 * lane));
            qraw[r] = (!half || (lane >> 5) == sl / r_half) ? w : 0u;
        }
    }
    // The A operands are q * 2^(10-2m) as f16, up to q * 2^6, and partly scaled up again below: large query elements would
    // not fit.  When the wave's largest |q| reaches 2^7 the whole query is taken divided by a power of two
    // (exact) that brings it below, and the softmax scale carries the factor back; 0 for ordinary queries.
    int q_down = 0;
    {
        float qa = 0.0f;
#pragma unroll
        for (int r = 0; r < NH; ++r)
            qa = fmaxf(qa, fmaxf(fabsf(__uint_as_float(qraw[r] << 16)), fabsf(__uint_as_float(qraw[r] & 0xFFFF0000u))));
        if (__builtin_expect(any_lane(qa >= 128.0f), 0)) {
            float m4[4] = {qa, qa, qa, qa};
            wave_max4(m4);
            q_down = min(static_cast<int>((__float_as_uint(m4[0]) >> 23) & 0xFFu) - 127 - 6, 100);
        }
    }
    if constexpr (LONG && !ANY) {
        if (__builtin_expect(q_down >= HUGE_Q_DOWN, 0)) goto other_form;
    }
    const float q_mul = __uint_as_float(static_cast<uint32_t>(127 - q_down) << 23);      // 2^-q_down
    // (uniform: kept in a scalar register, like the argument it stands for)
    const float sm_scale = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(
        a.sm_scale * __uint_as_float(static_cast<uint32_t>(127 + q_down) << 23))));
    if (__builtin_expect(q_down != 0, 0)) {
        // the per-channel copies too (thresholds and exact residuals below then need no factor of their own)
#pragma unroll
        for (int r = 0; r < NH; ++r) {
            const float lo = __uint_as_float(qraw[r] << 16) * q_mul, hi = __uint_as_float(qraw[r] & 0xFFFF0000u) * q_mul;
            qraw[r] = (__float_as_uint(lo) >> 16) | (__float_as_uint(hi) & 0xFFFF0000u);
        }
    }
    // The 32-token groups (64-token pieces of longer ones) are dealt out evenly: every split takes G/S of them and
    // the first G%S splits one more, so no two splits differ by more than one group and none is empty while
    // G >= S.  (One 32-bit division; the combine weighs the states by their lse, -inf for an
    // empty split, so it need not know this rule.)
    if (L < 0) { L = 0; report_table_range(a.err, true); }      // a negative length: nothing packed, reported
    const uint32_t G = static_cast<uint32_t>(L + (1 << UNIT_SH) - 1) >> UNIT_SH;
    const uint32_t g_each = G / S, g_more = G - g_each * S;
    const uint32_t g_first = static_cast<uint32_t>(sp) * g_each + min(static_cast<uint32_t>(sp), g_more);
    const uint32_t g_count = g_each + (static_cast<uint32_t>(sp) < g_more ? 1u : 0u);
    const int n_begin = static_cast<int>(g_first << UNIT_SH);
    const int n_end = min(static_cast<int>((g_first + g_count) << UNIT_SH), L);

    if (n_begin >= n_end) {       // an empty split: the state of nothing attended
        for (int r = 0; r < heads; ++r) {
            float* dst = a.al + b * a.al_b + (int64_t)(qh0 + r) * a.al_h + (int64_t)sp * a.al_s;
            dst[lane] = 0.0f;
            if (!half) dst[64 + lane] = 0.0f;
            if (lane == 0) a.sl[b * a.sl_b + (int64_t)(qh0 + r) * a.sl_h + (int64_t)sp * a.sl_s] = -INFINITY;
        }
        return;
    }

    // ---- addressing ---------------------------------------------------------------------------
    const uint32_t row_bytes = (uint32_t)Hkv * 32u;          // of a code row (k_base, v_main): below 2^24
    const int last = n_end - 1;
    const int ps_sh = __ffs(a.ps) - 1, ps_mask = a.ps - 1;
    const int tsh = a.i64 ? 3 : 2;
    const int tok_off = (a.gbase << GT_SH) + a.off;
    const char* const rt_b = static_cast<const char*>(a.rt) + ((b * a.rt_s) << tsh);
    const char* const rg_b = static_cast<const char*>(a.rg) + ((b * a.rg_s + a.gbase) << tsh);
    const uint8_t* const kb_head = a.k_base + kvh * 32;
    const uint8_t* const vb_head = a.v_main + kvh * 32;
    const int vv_sh = !LONG || a.gc == 32 ? 2 : a.gc == 64 ? 1 : 0;     // log2 of the V vectors per token
    const int8_t* const vs_head = a.v_scale + (kvh << vv_sh);
    const uint16_t* const vz_head = a.v_zp + (kvh << vv_sh);

    int pg1, ps1, gsl[NG];
    auto fetch_tables = [&](int n) {
        const int p = min(n + lane, last) + tok_off;
        pg1 = *reinterpret_cast<const int*>(rt_b + ((uint32_t)(p >> ps_sh) << tsh));
        ps1 = p & ps_mask;
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int gi = min((n + 32 * g) >> GT_SH, last >> GT_SH);
            gsl[g] = *reinterpret_cast<const int*>(rg_b + ((uint32_t)gi << tsh));
        }
    };
    bool bad_id = false;            // a table entry outside the planes was seen (and clamped)
    bool over_step = false;         // a K or V step above 2^MAX_STEP_EXP was seen (and held there); wave-uniform
    // Every plane this kernel is launched on is smaller than 4 GiB (the launcher sends larger ones to the
    // kernel in ommx_decode.hip), so a row or a group is a scalar plane pointer plus a 32-bit byte offset:
    // no 64-bit address arithmetic in the loop.
    u32x4 kr[2], vr[2];
    u32x2 vzp;
    uint32_t vsc, vro;
    auto at = [](const void* base, uint32_t byte_off) { return static_cast<const char*>(base) + byte_off; };
    auto fetch_k = [&]() {          // K code row of this lane's token; remembers the row offset for fetch_v
        pg1 = clamp_id(pg1, a.n_pages, bad_id);
        vro = __umul24(static_cast<uint32_t>((pg1 << ps_sh) + ps1), row_bytes);
        kr[0] = *reinterpret_cast<const u32x4*>(at(kb_head, vro));
        kr[1] = *reinterpret_cast<const u32x4*>(at(kb_head, vro + 16));
    };
    auto fetch_v = [&]() {          // a row of v_scale is an eighth, a row of v_zp a quarter of a code row
        vr[0] = *reinterpret_cast<const u32x4*>(at(vb_head, vro));
        vr[1] = *reinterpret_cast<const u32x4*>(at(vb_head, vro + 16));
        if (vv_sh == 2) {
            vsc = *reinterpret_cast<const uint32_t*>(at(vs_head, vro >> 3));
            vzp = *reinterpret_cast<const u32x2*>(at(vz_head, vro >> 2));
        } else if (vv_sh == 1) {        // (spread over the four 32-channel quarters where they are used)
            vsc = *reinterpret_cast<const uint16_t*>(at(vs_head, vro >> 4));
            vzp[0] = *reinterpret_cast<const uint32_t*>(at(vz_head, vro >> 3));
        } else {
            vsc = *reinterpret_cast<const uint8_t*>(at(vs_head, vro >> 5));
            vzp[0] = *reinterpret_cast<const uint16_t*>(at(vz_head, vro >> 4));
        }
    };
    // channel pair (2*lane, 2*lane+1) parameters of both groups
    uint32_t g_sc[NG], g_zp[NG], g_ms[NG] = {}, g_mc[NG] = {};
    u32x2 g_bm[NG], g_ov[NG];
    uint32_t g_bx[NG] = {};
    // 10 outliers: 18 index bytes and 10 nibble bytes per lane start at a multiple of 2; the aligned dwords that
    // cover them are loaded and shifted into place when they are used
    uint32_t g_ix10[5] = {}, g_ov10[3] = {};
    const uint32_t kvh_s = __builtin_amdgcn_readfirstlane(kvh);
    auto fetch_params_g = [&](int g) {
        // (the lane number goes through an opaque copy: otherwise plane pointer + lane offset is kept
        // as a 64-bit register pair per plane across the loop, twelve registers the QK phase lacks;
        // this way the loads take a scalar base and a 32-bit lane offset)
        uint32_t lane_b = lane;
        asm volatile("" : "+v"(lane_b));
        const uint32_t gs = __builtin_amdgcn_readfirstlane(clamp_id(gsl[g], a.n_gslots, bad_id));
        const uint32_t gidx = (gs * static_cast<uint32_t>(Hkv) + kvh_s) * D;      // first channel of the group, in elements
        const uint32_t ch = gidx + 2 * lane_b;                                    // this lane's channel pair
        g_sc[g] = *reinterpret_cast<const uint16_t*>(at(a.k_scale, ch));
        g_zp[g] = *reinterpret_cast<const uint32_t*>(at(a.k_zp, 2 * ch));
        if (OWN_MAP) {
            g_ms[g] = *reinterpret_cast<const uint32_t*>(at(a.k_ms, 2 * ch));
            g_mc[g] = *reinterpret_cast<const uint32_t*>(at(a.k_mc, 2 * ch));
        }
        if constexpr (KMAX == 10) {
            const uint32_t* ixp = reinterpret_cast<const uint32_t*>(at(a.k_obmp, 9 * gidx + ((18 * lane_b) & ~3u)));
#pragma unroll
            for (int i = 0; i < 5; ++i) g_ix10[i] = ixp[i];
            const uint32_t* ovp = reinterpret_cast<const uint32_t*>(at(a.k_oval, 5 * gidx + ((10 * lane_b) & ~3u)));
#pragma unroll
            for (int i = 0; i < 3; ++i) g_ov10[i] = ovp[i];
        } else if constexpr (IDX == 0) {
            g_bm[g] = *reinterpret_cast<const u32x2*>(at(a.k_obmp, 4 * ch));
        } else {
            const uint32_t* ixp = reinterpret_cast<const uint32_t*>(at(a.k_obmp, 6 * ch));
            g_bm[g] = u32x2{ixp[0], ixp[1]};
            g_bx[g] = ixp[2];
        }
        if constexpr (KMAX == 10) {
        } else if constexpr (!GEN) {
            // 3 nibble bytes per channel: the two dwords that hold the pair's six bytes
            const uint32_t* ovp = reinterpret_cast<const uint32_t*>(at(a.k_oval, 3 * gidx + 4 * ((3 * lane_b) / 2)));
            g_ov[g] = u32x2{ovp[0], ovp[1]};
        } else {
            // (kout + 1) / 2 bytes per channel, two channels per lane: the dword(s) that hold them
            const uint32_t kb = static_cast<uint32_t>(kout + 1) >> 1;
            const uint32_t* ovp = reinterpret_cast<const uint32_t*>(at(a.k_oval, gidx * kb + ((2 * kb * lane_b) & ~3u)));
            g_ov[g][0] = ovp[0];
            g_ov[g][1] = kb > 2 ? ovp[1] : 0u;       // 1 or 2 bytes per channel: one dword holds the pair
        }
    };
    // The page and group ids of the first step are asked for here; what follows (the A operands) needs
    // none of it and runs while they are on their way.
    fetch_tables(n_begin);
    asm volatile("" ::: "memory");

    // ---- A operand of QK: q * 2^(10-2m) of head j % 4 for this lane's 32-channel quarter, f16, in
    // pair order: k=(ks,kq,r) <-> channel 32kq + 16(ks/2) + 4(ks%2) + r/2 + 8(r%2).  The base codes,
    // the outlier tile and the bias columns all use this one operand (the tile and the zero points
    // are stored divided by the channel's 2^(10-2m)).
    u32x4 aq[4];
    u32x4 aq_any[ANY ? 4 : 1];            // ANY: q itself as bf16, divided like the f16 operand
    {
        auto q_at = [&](int c) {
            return __uint_as_float((c & 1) ? (qw[c >> 1] & 0xFFFF0000u) : (qw[c >> 1] << 16));
        };
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) {
                const int cl = 16 * (ks >> 1) + 4 * (ks & 1) + rr;
                const float qs = static_cast<float>(1 << (10 - 2 * k_pos<LONG>(4 * (ks & 1) + rr))) * q_mul;
                aq[ks][rr] = pack_f16x2(qs * q_at(cl), qs * q_at(cl + 8));
                if constexpr (ANY)
                    aq_any[ks][rr] = __builtin_amdgcn_perm(__float_as_uint(q_mul * q_at(cl + 8)), __float_as_uint(q_mul * q_at(cl)), 0x07060302u);
            }
        }
    }
    // The first step's data is asked for as soon as the page and group ids are here; clearing LDS, the
    // accumulators and the lane constants need none of it and run while it is on its way (the A operands
    // above ran while the ids were; with the clearing of LDS up there as well the request goes out late
    // again: 31.0 against 29.8 us at batch 1, 64K).  The instantiation with the most registers in flight (position
    // streams with their own outlier map, 4 heads) asks after the constants instead: with the loaded rows
    // live across them it would spill.
    constexpr bool FETCH_FIRST = !(IDX == 1 && OWN_MAP && NH == 4);
    auto first_fetch = [&]() {
        // in the order the first step needs them: K rows, the group parameters, then V
        fetch_k();
#pragma unroll
        for (int g = 0; g < NG; ++g) fetch_params_g(g);
        fetch_v();
        fetch_tables(n_begin + 64);
        asm volatile("" ::: "memory");
    };
    if constexpr (FETCH_FIRST) first_fetch();

    // ---- LDS that starts out constant: zero tile, zero corrections, the zero and one rows ----
    {
        u32x4* p = reinterpret_cast<u32x4*>(sm + OFF_TILE);
        for (int i = lane; i < 32 * TILE_ROW / 16; i += 64) p[i] = u32x4{0, 0, 0, 0};
        for (int i = lane; i < (LONG ? 16 : 8) * NH; i += 64) reinterpret_cast<u32x4*>(sm + OFF_LC)[i] = u32x4{0, 0, 0, 0};
        if (lane < 16) reinterpret_cast<u32x4*>(sm + OFF_ZERO)[lane] =
            lane < 8 ? u32x4{0, 0, 0, 0} : u32x4{0x3C003C00u, 0x3C003C00u, 0x3C003C00u, 0x3C003C00u};
    }

    // output accumulators: with 4 heads the 16 columns are 4 replicas of the heads and replica x takes
    // the channel blocks Y = x, x + 4 (two accumulators); with 8 heads they are 2 replicas and replica x
    // takes Y = x, x + 2, x + 4, x + 6 (four)
    f32x4 acc[NH / 2];
#pragma unroll
    for (int i = 0; i < NH / 2; ++i) acc[i] = f32x4{0, 0, 0, 0};
    f32x4 accz = {0, 0, 0, 0};
    float m_run[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) m_run[r] = -INFINITY;


    auto q_of = [&](int u, int r) { return __uint_as_float(u ? (qraw[r] & 0xFFFF0000u) : (qraw[r] << 16)); };
    // ---- lane constants of the loop ------------------------------------------------------------
    // channel pass: lane = channels c0 = 2*lane, c0 + 1
    const uint32_t c0 = 2u * lane;
    const uint32_t y0 = c0 & 15u;
    // halfword slot of channel c0 in the pair-ordered arrays; channel c0 + 1 sits two slots on
    const uint32_t hw0 = ((c0 >> 4) * 8u + (y0 & 7u)) * 2u + (y0 >> 3);
    // 2^-(10-2m) of the two channels: what their zero points and tile entries are scaled by
    const float cs0 = 1.0f / static_cast<float>(1 << (10 - 2 * k_pos<LONG>(int(y0 & 7u))));
    const float cs1 = 1.0f / static_cast<float>(1 << (10 - 2 * k_pos<LONG>(int((y0 + 1u) & 7u))));
    // per channel: the |tile entry| from which its f16 rounding matters (infinite for q = 0)
    float big_thr[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        float qm = 0.0f;
#pragma unroll
        for (int r = 0; r < NH; ++r)
            qm = fmaxf(qm, fabsf(__uint_as_float(u ? (qraw[r] & 0xFFFF0000u) : (qraw[r] << 16))));
        big_thr[u] = ((GEN || HALF ? (kout < 6 ? 0.5f : 0.75f) : 1.0f) * BIG_DELTA * 16.0f * BIG_DELTA_SM_SCALE) * (u ? cs1 : cs0) *
                     __builtin_amdgcn_rcpf(qm * sm_scale);
        if (LONG) big_thr[u] = fminf(big_thr[u], MAX_F16);     // (what no f16 holds is looked at whatever q is)
    }
    const uint32_t kt_lane = OFF_KT + (c0 >> 2);                   // code byte of the channel pair (4 channels a byte), row 0
    const uint32_t code_bits = 3u << (2u * (c0 & 3u));            // of channel c0's code in that byte; c0 + 1 sits two bits on
    // A code is taken where it lies in its byte, as the bits of a subnormal f16, 2^-24 each: a mask and one mixed multiply-add, in
    // the place of a shift, a conversion and a multiply-add.  Exact, as long as its step times 2^24 is an fp32 number; ANY, where
    // steps of every size come by, takes the masked byte as a number.  This is the exponent of the unit that it counts.
    auto code_unit = [&](int u) { return (ANY ? 0 : 24) - ((lane & 1) ? 4 : 0) - 2 * u; };
    const uint32_t kbytes = static_cast<uint32_t>(kout + 1) >> 1;            // nibble bytes per channel
    const uint32_t nib_sh = 8u * ((2u * kbytes * lane) & 3u);
    const uint32_t nib_at = (lane & 1) ? 0x0C040302u : 0x0C020100u;          // 6 outliers: the bytes of channel c0's nibbles (c0 + 1: three on)
    const float c2 = sm_scale * 1.4426950408889634f;
    if constexpr (!FETCH_FIRST) first_fetch();

    for (int n0 = n_begin; n0 < n_end; n0 += 64) {
        const bool more = n0 + 64 < n_end;
        const bool g1_live = n0 + 32 < n_end;
        {   // waves sharing a SIMD should finish together: the one with more work left goes first
            const int left = (n_end - n0 + 63) >> 6;
            if (left >= 4) __builtin_amdgcn_s_setprio(3);
            else if (left == 3) __builtin_amdgcn_s_setprio(2);
            else if (left == 2) __builtin_amdgcn_s_setprio(1);
            else __builtin_amdgcn_s_setprio(0);
        }

        // ------------------------------------------------------------------ stage K
        bool exact_step = false;                // some step of these 64 tokens is 2^EXACT_STEP_EXP or more (wave-uniform)
        // LONG: exponents counted from MIN_STEP_EXP, unsigned (smaller ones become the largest numbers, from BELOW on), and
        // what the zero points are too large by; either out of bounds takes the branch of an exact step, which looks closer
        typedef unsigned short u16x2e __attribute__((ext_vector_type(2)));
        u16x2e e_from = {0, 0}, zp_over = {0, 0};
        uint32_t dead[2] = {0, 0};              // code bits, in the lane's K operands, of channels with a step below the range
        constexpr uint16_t EXACT = (EXACT_STEP_EXP - MIN_STEP_EXP) * 256, MOST = (MAX_STEP_EXP - MIN_STEP_EXP) * 256,
                           BELOW = (256 - 128 - MIN_STEP_EXP) * 256;
        if constexpr (LONG && !ANY) {
            e_from = __builtin_bit_cast(u16x2e, __builtin_amdgcn_perm(0u, g_sc[0], 0x010C000Cu)) + static_cast<uint16_t>(-MIN_STEP_EXP * 256);
            zp_over = __builtin_elementwise_sub_sat(__builtin_bit_cast(u16x2e, g_zp[0] & 0x7FFF7FFFu),
                                                    u16x2e{ANY_ZP_BF16 - 1, ANY_ZP_BF16 - 1});
            exact_step = any_lane((e_from[0] > e_from[1] ? e_from[0] : e_from[1]) >= EXACT || __builtin_bit_cast(uint32_t, zp_over) != 0) ||
                         q_down != 0;
        } else if constexpr (!ANY) {
            typedef short s16x2e __attribute__((ext_vector_type(2)));
            const s16x2e top2 = __builtin_elementwise_max(
                __builtin_bit_cast(s16x2e, __builtin_amdgcn_perm(0u, g_sc[0], 0x010C000Cu)),
                __builtin_bit_cast(s16x2e, __builtin_amdgcn_perm(0u, g_sc[NG - 1], 0x010C000Cu)));
            const short e_top = top2[0] > top2[1] ? top2[0] : top2[1];
            // (a scaled-down query means operands near the top of f16: the same cancellation, the same remedy)
            // (not any_lane: with this test in a scalar register up to 16 vector registers are spilled)
            exact_step = __any(e_top >= EXACT_STEP_EXP * 256) != 0 || q_down != 0;
            if (__builtin_expect(exact_step, 0)) {
                over_step |= __any(e_top > MAX_STEP_EXP * 256) != 0;
                // (the walk below takes such a step times 2^24, past the largest fp32 if it is not held here: far outside f16, as it was)
#pragma unroll
                for (int g = 0; g < NG; ++g) {
                    const uint32_t held = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(
                        __builtin_bit_cast(s16x2e, __builtin_amdgcn_perm(0u, g_sc[g], 0x010C000Cu)), s16x2e{CODE_STEP_EXP * 256, CODE_STEP_EXP * 256}));
                    g_sc[g] = __builtin_amdgcn_perm(0u, held, 0x0C0C0301u);
                }
            }
        }
        {
            u32x2* krow = reinterpret_cast<u32x2*>(sm + OFF_KT + lane * KT_ROW);
            krow[0] = u32x2{kr[0][0], kr[0][1]};
            krow[1] = u32x2{kr[0][2], kr[0][3]};
            krow[2] = u32x2{kr[1][0], kr[1][1]};
            krow[3] = u32x2{kr[1][2], kr[1][3]};
            uint16_t* mg = reinterpret_cast<uint16_t*>(sm + OFF_MAG) + hw0;
            uint16_t* zp = reinterpret_cast<uint16_t*>(sm + OFF_ZPP) + hw0;
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                // f16 2^e of both channels: (e + 15) << 10 per half, e a signed byte held at -15 or
                // above (a step below 2^-14 is immaterial next to the f16 operands of the others)
                const uint32_t e2 = __builtin_amdgcn_perm(0u, g_sc[g], 0x010C000Cu);       // (e1 << 8, e0 << 8)
                typedef short s16x2 __attribute__((ext_vector_type(2)));
                typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
                constexpr short LEAST = (LONG ? MIN_STEP_EXP : -15) * 256;
                const s16x2 ec = __builtin_elementwise_min(
                    __builtin_elementwise_max(__builtin_bit_cast(s16x2, e2), s16x2{LEAST, LEAST}),
                    s16x2{MAX_STEP_EXP * 256, MAX_STEP_EXP * 256});
                uint32_t m2 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2, ec) * u16x2{4, 4} + u16x2{0x3C00, 0x3C00});
                if constexpr (ANY) {       // bf16 2^e
                    const int e0 = static_cast<int8_t>(g_sc[g] & 0xFFu), e1 = static_cast<int8_t>((g_sc[g] >> 8) & 0xFFu);
                    m2 = pk_u16(static_cast<uint32_t>(e0 + 127) << 7, static_cast<uint32_t>(e1 + 127) << 7);
                }
                mg[g * 128] = static_cast<uint16_t>(m2);
                mg[g * 128 + 2] = static_cast<uint16_t>(m2 >> 16);
                // zero points over the channel's A scale (exact: a power of two), f16; ANY: as they are
                const uint32_t z2 = ANY ? g_zp[g] : pack_f16x2(cs0 * __uint_as_float(g_zp[g] << 16),
                                                               cs1 * __uint_as_float(g_zp[g] & 0xFFFF0000u));
                zp[g * 128] = static_cast<uint16_t>(z2);
                zp[g * 128 + 2] = static_cast<uint16_t>(z2 >> 16);
            }
        }
        lds_fence();
        if (more) fetch_k();

        // ------------------------------------------------------------------ QK
        // 4 heads: the lane keeps the logits of its own token n0 + lane (one 16-token block of one group);
        // 8 heads: rows 4kq..4kq+3 are heads 4(kq & 1)..+3, and the lane keeps those four heads of token
        // 16(kq >> 1) + j of either group
        f32x4 dsel[NH / 4];
#pragma unroll
        for (int i = 0; i < NH / 4; ++i) dsel[i] = f32x4{0, 0, 0, 0};
        // Longer groups: both halves of the step lie in one group, whose outliers are walked once: what an outlier adds, as f16, and
        // the tile row it goes to in half 0 (as an offset; half 1 lies 32 rows on, and what lies in neither half past both).
        // Each half then takes the scatter alone.  Walked anew for every half, as before, the positions, code reads and entries
        // are formed twice; vector instructions are what these kernels are nearest to a limit of.  Whole call, 32 requests of 1
        // to 16 K: 64 x 64 with six outliers 105.8 -> 99.2 us, 128 x 128 with ten 125.5 -> 113.2; 4 of 2 to 20 K of those
        // 31.3 -> 28.9, 64 K alone 37.1 -> 35.2, 16 of 2 to 16 K with 64 q heads 78.5 -> 71.9.
        uint32_t l_at[LONG ? 2 : 1][KMAX];
        uint16_t l_e[LONG ? 2 : 1][KMAX];
        bool l_res = false;
        constexpr uint32_t HALF_ROWS = 32u * TILE_ROW;
        if constexpr (LONG) {
            float dls[2][KMAX];
            auto walk = [&](auto U) {
                constexpr int u = decltype(U)::value;
                // index bits and levels of the channel; 10 outliers: the lane's bytes start 0 or 2 bytes into the loaded dwords
                uint32_t ixw[3] = {0, 0, 0}, o0, o1 = 0;
                if constexpr (KMAX == 10) {
                    const uint32_t sh = ((lane & 1) ? 16u : 0u) + (u ? 8u : 0u);
#pragma unroll
                    for (int i = 0; i < 3; ++i)
                        ixw[i] = (i == 2 && u) ? g_ix10[4] >> sh : __builtin_amdgcn_alignbit(g_ix10[i + 1 + 2 * u], g_ix10[i + 2 * u], sh);
                    o0 = __builtin_amdgcn_alignbit(g_ov10[1 + u], g_ov10[u], sh);
                    o1 = u ? g_ov10[2] >> sh : __builtin_amdgcn_alignbit(g_ov10[2], g_ov10[1], sh);
                } else {
                    ixw[0] = u ? __builtin_amdgcn_alignbit(g_bx[0], g_bm[0][1], 16) : g_bm[0][0];
                    ixw[1] = u ? (g_bx[0] >> 16) : g_bm[0][1];
                    o0 = __builtin_amdgcn_perm(g_ov[0][1], g_ov[0][0], nib_at + (u ? 0x030303u : 0u));
                }
                // 128 tokens: the upper bit of every position flipped in the second piece, so that those of the piece read below 64
                if (GTS == 2 && (n0 & 64)) {
#pragma unroll
                    for (int i = 0; i < 3; ++i) {
                        uint32_t two = 0;
                        for (int s7 = 0; s7 < KMAX; ++s7)
                            if ((7 * s7 + 6) >> 5 == i) two |= 1u << ((7 * s7 + 6) & 31);
                        ixw[i] ^= two;
                    }
                }
                uint32_t cb[KMAX];
#pragma unroll
                for (int sidx = 0; sidx < KMAX; ++sidx) {
                    constexpr uint32_t PM = (1u << GT_SH) - 1;
                    const int bit = 7 * sidx, wi = bit >> 5, bo = bit & 31;
                    const uint32_t f = (bo + GT_SH <= 32 ? (ixw[wi] >> bo) : __builtin_amdgcn_alignbit(ixw[wi < 2 ? wi + 1 : 2], ixw[wi], bo)) & PM;
                    const uint32_t pos = GTS == 2 ? min(f, 64u) : f;
                    l_at[u][sidx] = pos * TILE_ROW;
                    cb[sidx] = *(sm + kt_lane + pos * KT_ROW);        // (of a row past the 64 nothing is used)
                }
                const float zp = __uint_as_float(u ? (g_zp[0] & 0xFFFF0000u) : (g_zp[0] << 16));
                const int e = static_cast<int8_t>((g_sc[0] >> (8 * u)) & 0xFFu);
                // in units of the channel's A scale, as in the walk of 32-token groups below
                const float cs = u ? cs1 : cs0;
                const float code_step = __builtin_ldexpf(cs, e + code_unit(u));
                float a1, b1 = 0.0f;
                if (OWN_MAP) {
                    a1 = cs * __builtin_amdgcn_rcpf(__uint_as_float(u ? (g_ms[0] & 0xFFFF0000u) : (g_ms[0] << 16)));
                    b1 = cs * (__uint_as_float(u ? (g_mc[0] & 0xFFFF0000u) : (g_mc[0] << 16)) - zp);
                } else {
                    a1 = __builtin_ldexpf(cs, e);
                }
                float lv[10];
                const f32x2 l01 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(o0, 1.0f, 0);
                const f32x2 l23 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(o0, 1.0f, 1);
                const f32x2 l45 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(o0, 1.0f, 2);
                lv[0] = l01[0]; lv[1] = l01[1]; lv[2] = l23[0]; lv[3] = l23[1]; lv[4] = l45[0]; lv[5] = l45[1];
                if constexpr (KMAX == 10) {
                    const f32x2 l67 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(o0, 1.0f, 3);
                    const f32x2 l89 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(o1, 1.0f, 0);
                    lv[6] = l67[0]; lv[7] = l67[1]; lv[8] = l89[0]; lv[9] = l89[1];
                }
                float dl_max = 0.0f;
#pragma unroll
                for (int sidx = 0; sidx < KMAX; ++sidx) {
                    const uint32_t code = cb[sidx] & (code_bits << 2 * u);
                    float dl = fmaf(ANY ? -static_cast<float>(code) : -f16_bits(code), code_step, fmaf(lv[sidx], a1, b1));
                    // (the entry as a value of its own: rounded to f16 here exactly as the residual pass rounds it)
                    asm("" : "+v"(dl));
                    dls[u][sidx] = dl;
                    // (ANY: the tile takes the largest f16, the logits the rest)
                    l_e[u][sidx] = __builtin_bit_cast(uint16_t, static_cast<_Float16>(
                        ANY && fabsf(dl) > MAX_F16 ? copysignf(MAX_F16, dl) : dl));
                    dl_max = fmaxf(dl_max, GTS == 1 || l_at[u][sidx] < 2 * HALF_ROWS ? fabsf(dl) : 0.0f);
                }
                return (ANY && q_down >= HUGE_Q_DOWN) || any_lane(dl_max >= big_thr[u]);
            };
            // Entries of the step whose f16 rounding matters add what the rounding dropped to the logits, exactly.
            auto residuals = [&](auto U) {
                constexpr int u = decltype(U)::value;
                const float un = __builtin_amdgcn_rcpf(u ? cs1 : cs0);
                float* lc = reinterpret_cast<float*>(sm + OFF_LC);
#pragma unroll
                for (int sidx = 0; sidx < KMAX; ++sidx) {
                    const float dl = dls[u][sidx], hi = static_cast<float>(__builtin_bit_cast(_Float16, l_e[u][sidx]));
                    bool matters = fabsf(dl) >= big_thr[u];
                    if constexpr (ANY) matters |= q_down >= HUGE_Q_DOWN && fabsf(dl) < MIN_F16 && dl != hi;
                    if (matters && (GTS == 1 || l_at[u][sidx] < 2 * HALF_ROWS)) {
                        const float lo = (dl - hi) * un;
                        float* at_pos = lc + l_at[u][sidx] / TILE_ROW * NH;
#pragma unroll
                        for (int r = 0; r < NH; ++r)
                            __hip_atomic_fetch_add(at_pos + r, lo * q_of(u, r), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
                    }
                }
            };
            const bool res0 = walk(std::integral_constant<int, 0>{});
            if (res0) residuals(std::integral_constant<int, 0>{});
            const bool res1 = walk(std::integral_constant<int, 1>{});
            if (res1) residuals(std::integral_constant<int, 1>{});
            l_res = res0 || res1;
            if (more) fetch_params_g(0);
        }
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            if (g == 1 && !g1_live) break;
            const int pg = LONG ? 0 : g;           // the group's parameter set
            float* lc = reinterpret_cast<float*>(sm + OFF_LC) + (LONG ? 32 * NH * g : 0);
            bool res_any = l_res;
            if constexpr (LONG) {
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int sidx = 0; sidx < KMAX; ++sidx)
                        *reinterpret_cast<uint16_t*>(sm + OFF_TILE + 2 * hw0 + 4 * u + min(l_at[u][sidx] - g * HALF_ROWS, HALF_ROWS)) = l_e[u][sidx];
            } else {
            // The channel pass of a group in two halves, so that the code bytes of both channels are on their
            // way before either channel's entries need them: positions and code reads, then entries and scatter.
            // The base MFMA takes every position of the K rows as it is stored; the tile entry of an
            // outlier is what is missing on top of its stored 2-bit code, which the lane looks up
            // in the staged K rows (a byte read per outlier; the packer's code of an outlier is the
            // clamped 0 or 3 nearly always, so the entry is small).
            auto walk_read = [&](auto U, int (&pos)[KMAX], uint32_t (&cb)[KMAX]) {
                constexpr int u = decltype(U)::value;
                uint32_t bm = 0, ix_lo = 0, ix_hi = 0;
                if constexpr (IDX == 0) {
                    bm = g_bm[pg][u];
                } else {
                    ix_lo = u ? __builtin_amdgcn_alignbit(g_bx[pg], g_bm[pg][1], 16) : g_bm[pg][0];
                    ix_hi = u ? (g_bx[pg] >> 16) : g_bm[pg][1];
                }
                const uint8_t* kt = sm + kt_lane + g * 32 * KT_ROW;
#pragma unroll
                for (int sidx = 0; sidx < KMAX; ++sidx) {
                    if constexpr (IDX == 0) {
                        pos[sidx] = lowest_bit(bm);
                        if (sidx < KMAX - 1) bm = without_bit(bm, pos[sidx]);
                    } else {
                        pos[sidx] = sidx < 4 ? ((ix_lo >> (7 * sidx)) & 31)
                                  : sidx == 4 ? (__builtin_amdgcn_alignbit(ix_hi, ix_lo, 28) & 31)
                                              : ((ix_hi >> 3) & 31);
                    }
                    cb[sidx] = kt[pos[sidx] * KT_ROW];
                }
            };
            auto walk_write = [&](auto U, const int (&pos)[KMAX], const uint32_t (&cb)[KMAX], float (&dls)[KMAX]) {
                constexpr int u = decltype(U)::value;
                const float zp = __uint_as_float(u ? (g_zp[pg] & 0xFFFF0000u) : (g_zp[pg] << 16));
                const int e = static_cast<int8_t>((g_sc[pg] >> (8 * u)) & 0xFFu);
                // everything below is in units of the channel's A scale: tile entry =
                // (outlier - zp - code * 2^e) / 2^(10-2m) = level * a1 + b1 less the code's step times the code
                const float cs = u ? cs1 : cs0;
                // (With codes by two instructions, positions by two instead of three, one test a channel for residuals and nibbles
                // by one permutation the pass over a group's outliers is 126 vector instructions, 157 before: 64 K 31.4 -> 30.8 us,
                // 8 x 32 K with 64 q heads 103.5 -> 102.4, 32 of 1 to 16 K with position streams 100.3 -> 98.7.)
                const float code_step = __builtin_ldexpf(cs, e + code_unit(u));
                float a1, b1;
                if (OWN_MAP) {
                    const float ms = __uint_as_float(u ? (g_ms[pg] & 0xFFFF0000u) : (g_ms[pg] << 16));
                    const float mc = __uint_as_float(u ? (g_mc[pg] & 0xFFFF0000u) : (g_mc[pg] << 16));
                    a1 = cs * __builtin_amdgcn_rcpf(ms);
                    b1 = cs * (mc - zp);
                } else {
                    a1 = __builtin_ldexpf(cs, e);
                    b1 = 0.0f;
                }
                float lv[8];
                uint32_t nib;
                if constexpr (GEN) nib = static_cast<uint32_t>(((static_cast<uint64_t>(g_ov[pg][1]) << 32) | g_ov[pg][0]) >> (nib_sh + 8 * kbytes * u));
                else nib = __builtin_amdgcn_perm(g_ov[pg][1], g_ov[pg][0], nib_at + (u ? 0x030303u : 0u));
                const f32x2 l01 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(nib, 1.0f, 0);
                const f32x2 l23 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(nib, 1.0f, 1);
                const f32x2 l45 = KMAX > 4 ? __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(nib, 1.0f, 2) : f32x2{0.0f, 0.0f};
                const f32x2 l67 = KMAX > 6 ? __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(nib, 1.0f, 3) : f32x2{0.0f, 0.0f};
                lv[0] = l01[0]; lv[1] = l01[1]; lv[2] = l23[0]; lv[3] = l23[1]; lv[4] = l45[0]; lv[5] = l45[1];
                lv[6] = l67[0]; lv[7] = l67[1];
                uint16_t* dt = reinterpret_cast<uint16_t*>(sm + OFF_TILE) + hw0 + 2 * u;      // pair order, like MAG
                float dl_max = 0.0f;
#pragma unroll
                for (int sidx = 0; sidx < KMAX; ++sidx) {
                    const float dl0 = fmaf(lv[sidx], a1, b1);
                    const uint32_t code = cb[sidx] & (code_bits << 2 * u);
                    float dl = fmaf(-f16_bits(code), code_step, dl0);
                    // (the entry as a value of its own: rounded to f16 here exactly as the residual pass rounds it)
                    asm("" : "+v"(dl));
                    dls[sidx] = dl;
                    if (GEN && sidx >= kout) continue;          // an unused slot (uniform): nothing to write
                    dt[pos[sidx] * (TILE_ROW / 2)] = __builtin_bit_cast(uint16_t, static_cast<_Float16>(dl));
                    dl_max = fmaxf(dl_max, fabsf(dl));
                }
                return dl_max;
            };
            // Entries whose f16 rounding matters add what the rounding dropped to the logits, exactly
            // (rare, and kept out of the walks so that both channels' walks run as one stretch of code:
            // their positions and entries are still at hand)
            auto residuals = [&](auto U, const int (&pos)[KMAX], const float (&dls)[KMAX]) {
                constexpr int u = decltype(U)::value;
                const float un = __builtin_amdgcn_rcpf(u ? cs1 : cs0);
#pragma unroll
                for (int sidx = 0; sidx < KMAX; ++sidx) {
                    if (GEN && sidx >= kout) continue;
                    const float dl = dls[sidx];
                    if (fabsf(dl) >= big_thr[u]) {
                        const float hi = static_cast<float>(static_cast<_Float16>(dl));
                        const float lo = (dl - hi) * un;
                        if constexpr (HALF && !PARTIAL) {
                            // (the lane's channels belong to one kv head of the pair: the other's queries read zero there, and half
                            // of the adds would add nothing.  At 64^-0.5 on a logit 8 slots a group have an entry to settle, against 2
                            // at head_dim 128; whole call, 2 requests of 12 K 19.9 -> 18.5 us, 8 of 8 K 27.2 -> 25.1, 16 of 2 to
                            // 16 K 48.8 -> 42.2)
#pragma unroll
                            for (int r = 0; r < NH / 2; ++r) {
                                const uint32_t w = qraw[r] | qraw[r + NH / 2];
                                __hip_atomic_fetch_add(lc + pos[sidx] * NH + (lane >> 5) * (NH / 2) + r,
                                                       lo * __uint_as_float(u ? (w & 0xFFFF0000u) : (w << 16)), __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_WAVEFRONT);
                            }
                        } else {
#pragma unroll
                            for (int r = 0; r < NH; ++r)
                                __hip_atomic_fetch_add(lc + pos[sidx] * NH + r, lo * q_of(u, r), __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_WAVEFRONT);
                        }
                    }
                }
            };
            int pos0[KMAX], pos1[KMAX];
            uint32_t cb0[KMAX], cb1[KMAX];
            float dls0[KMAX], dls1[KMAX];
            // (the general form has fewer registers to spare: one channel after the other there)
            walk_read(std::integral_constant<int, 0>{}, pos0, cb0);
            if constexpr (!GEN) walk_read(std::integral_constant<int, 1>{}, pos1, cb1);
            const float dlm0 = walk_write(std::integral_constant<int, 0>{}, pos0, cb0, dls0);
            if constexpr (GEN) walk_read(std::integral_constant<int, 1>{}, pos1, cb1);
            const float dlm1 = walk_write(std::integral_constant<int, 1>{}, pos1, cb1, dls1);
            const bool res0 = any_lane(dlm0 >= big_thr[0]), res1 = any_lane(dlm1 >= big_thr[1]);
            res_any = res0 || res1;
            if (__builtin_expect(res0, 0)) residuals(std::integral_constant<int, 0>{}, pos0, dls0);
            if (__builtin_expect(res1, 0)) residuals(std::integral_constant<int, 1>{}, pos1, dls1);
            }
            lds_fence();
            if (more && !LONG) fetch_params_g(pg);
            // both 16-token blocks of the group go through the eight k-steps together (two independent
            // accumulation chains): tile rows (read, clear), then the base codes
            f32x4 d[2] = {f32x4{0, 0, 0, 0}, f32x4{0, 0, 0, 0}};
            u32x2 kw[2];
#pragma unroll
            for (int t2 = 0; t2 < 2; ++t2)
                kw[t2] = *reinterpret_cast<const u32x2*>(sm + OFF_KT + (16 * (2 * g + t2) + j) * KT_ROW + 8 * kq);
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
                for (int t2 = 0; t2 < 2; ++t2) {
                    u32x4* row = reinterpret_cast<u32x4*>(sm + OFF_TILE + (16 * t2 + j) * TILE_ROW + 64 * kq);
                    const u32x4 bt = row[ks];
                    row[ks] = u32x4{0, 0, 0, 0};
                    d[t2] = mfma_f16(aq[ks], bt, d[t2]);
                }
            }
            const u32x4* mg = reinterpret_cast<const u32x4*>(sm + OFF_MAG + pg * 256 + kq * 64);
            auto base_mfmas = [&](auto EX) {
                // EX: the operand without its constant, code * 2^(2m-10+e) = pattern - 2^e
                auto op = [&](uint32_t pat, uint32_t mag) {
                    if constexpr (!decltype(EX)::value) return pat;
                    else return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, pat) - __builtin_bit_cast(f16x2, mag));
                };
#pragma unroll
                for (int hf = 0; hf < 2; ++hf) {          // code dword: channels 16*hf .. 16*hf+15 of the quarter
                    uint32_t w[2], wu[2], wd[2];
#pragma unroll
                    for (int t2 = 0; t2 < 2; ++t2) { w[t2] = kw[t2][hf]; wu[t2] = w[t2] << (LONG ? 6 : 4); wd[t2] = w[t2] >> 6; }
                    const u32x4 ma = mg[2 * hf], mb = mg[2 * hf + 1];
#pragma unroll
                    for (int t2 = 0; t2 < 2; ++t2)
                        d[t2] = mfma_f16(aq[2 * hf], u32x4{op(k_pair<0, LONG>(w[t2], wu[t2], wd[t2], ma[0]), ma[0]), op(k_pair<1, LONG>(w[t2], wu[t2], wd[t2], ma[1]), ma[1]),
                                                           op(k_pair<2, LONG>(w[t2], wu[t2], wd[t2], ma[2]), ma[2]), op(k_pair<3, LONG>(w[t2], wu[t2], wd[t2], ma[3]), ma[3])}, d[t2]);
#pragma unroll
                    for (int t2 = 0; t2 < 2; ++t2)
                        d[t2] = mfma_f16(aq[2 * hf + 1], u32x4{op(k_pair<4, LONG>(w[t2], wu[t2], wd[t2], mb[0]), mb[0]), op(k_pair<5, LONG>(w[t2], wu[t2], wd[t2], mb[1]), mb[1]),
                                                               op(k_pair<6, LONG>(w[t2], wu[t2], wd[t2], mb[2]), mb[2]), op(k_pair<7, LONG>(w[t2], wu[t2], wd[t2], mb[3]), mb[3])}, d[t2]);
                }
            };
            if constexpr (ANY) {
                // code * 2^e as bf16
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) {
                    const u32x4 m = mg[ks];
#pragma unroll
                    for (int t2 = 0; t2 < 2; ++t2) {
                        u32x4 w;
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const uint32_t c2 = (kw[t2][ks >> 1] >> (2 * (4 * (ks & 1) + r))) & 0x00030003u;
                            w[r] = __builtin_amdgcn_perm(
                                __float_as_uint(static_cast<float>(c2 >> 16) * __uint_as_float(m[r] & 0xFFFF0000u)),
                                __float_as_uint(static_cast<float>(c2 & 0xFFFFu) * __uint_as_float(m[r] << 16)), 0x07060302u);
                        }
                        d[t2] = mfma_bf16(aq_any[ks], w, d[t2]);
                    }
                }
            } else if (__builtin_expect(exact_step, 0)) {
                if constexpr (LONG) {
                    if (g == 0) {
                        auto over = [&](uint16_t e) { return e > MOST && e < BELOW; };
                        if (any_lane(over(e_from[0]) || over(e_from[1]) || __builtin_bit_cast(uint32_t, zp_over) != 0)) goto other_form;
                        // a step below the range is harmless where all codes are zero (a channel that does not vary)
                        const uint64_t lo = __ballot(e_from[0] >= BELOW), hi = __ballot(e_from[1] >= BELOW);
                        if (lo | hi) {
#pragma unroll
                            for (int hf = 0; hf < 2; ++hf) {
                                auto spread = [&](uint64_t m) {      // eight lanes' bits, four apart
                                    uint32_t x = static_cast<uint32_t>(m >> (16 * kq + 8 * hf)) & 0xFFu;
                                    x = (x | x << 12) & 0x000F000Fu;
                                    x = (x | x << 6) & 0x03030303u;
                                    return (x | x << 3) & 0x11111111u;
                                };
                                dead[hf] = 3u * spread(lo) | 12u * spread(hi);
                            }
                        }
                    }
                    if (any_lane((((kw[0][0] | kw[1][0]) & dead[0]) | ((kw[0][1] | kw[1][1]) & dead[1])) != 0)) goto other_form;
                }
                base_mfmas(std::true_type{});
                // the bias MFMA must not take the constant out a second time: its 2^e column of this group reads zeros
                if (!LONG || g == 1 || !g1_live) {
                    lds_fence();
                    reinterpret_cast<uint32_t*>(sm + OFF_MAG + pg * 256)[lane] = 0u;
                }
            } else {
                base_mfmas(std::false_type{});
            }
            if constexpr (NH == 4) {
                // rows 4kq..4kq+3 of every result hold the four heads: the lane keeps its own token block
#pragma unroll
                for (int t2 = 0; t2 < 2; ++t2)
                    if (kq == 2 * g + t2 || (g == 0 && t2 == 0)) dsel[0] = d[t2];      // (group 1's lanes: theirs comes, or is not wanted)
                if (res_any) {       // exact residuals of this group's large deltas, then zero again
                    const f32x4 corr = *reinterpret_cast<const f32x4*>(lc + 4 * (lane & 31));
                    if ((kq >> 1) == g) dsel[0] += corr;
                    lds_fence();
                    *reinterpret_cast<u32x4*>(lc + 4 * (lane & 31)) = u32x4{0, 0, 0, 0};
                }
            } else {
                dsel[g] = (kq >> 1) ? d[1] : d[0];
                if (res_any) {
                    // the lane's token of this group, its four heads
                    dsel[g] += *reinterpret_cast<const f32x4*>(lc + 8 * (16 * (kq >> 1) + j) + 4 * (kq & 1));
                    lds_fence();
                    *reinterpret_cast<u32x4*>(lc + 4 * lane) = u32x4{0, 0, 0, 0};
                }
            }
            lds_fence();
        }
        // bias columns: 0 zp(g0) 1 zp(g1) 2 2^e(g0) 3 2^e(g1); other columns repeat them
        f32x4 dbias = {0, 0, 0, 0};
        {
            const int src = ANY && (j & 2) ? OFF_ZERO : ((j & 2) ? OFF_MAG : OFF_ZPP) + (LONG ? 0 : (j & 1) * 256) + kq * 64;
            const u32x4* bp = reinterpret_cast<const u32x4*>(sm + src);
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                if constexpr (ANY) dbias = mfma_bf16(aq_any[ks], bp[ks], dbias);
                else dbias = mfma_f16(aq[ks], bp[ks], dbias);
            }
        }
        if (more) fetch_tables(n0 + 128);
        lds_fence();

        // ------------------------------------------------------------------ stage V (over the K staging)
        uint32_t v_out = 0;                     // LONG: not zero: a V step of this token is outside the range
        {
            uint32_t* vt = reinterpret_cast<uint32_t*>(sm + OFF_VT) + lane;
#pragma unroll
            for (int c = 0; c < 8; ++c) vt[c * VT_COL] = vr[c >> 2][c & 3];
            typedef short s16x2 __attribute__((ext_vector_type(2)));
            typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
            if (LONG && vv_sh == 1) {
                vsc = __builtin_amdgcn_perm(0u, vsc, 0x01010000u);
                vzp = u32x2{__builtin_amdgcn_perm(0u, vzp[0], 0x01000100u), __builtin_amdgcn_perm(0u, vzp[0], 0x03020302u)};
            } else if (LONG && vv_sh == 0) {
                vsc = __builtin_amdgcn_perm(0u, vsc, 0x00000000u);
                vzp[0] = __builtin_amdgcn_perm(0u, vzp[0], 0x01000100u);
                vzp[1] = vzp[0];
            }
            // a V step above 2^MAX_STEP_EXP (a signed exponent byte of 16 or more) is held there and reported
            if constexpr (!LONG || ANY) {
                if (__builtin_expect(any_lane((((vsc & 0x7F7F7F7Fu) + 0x70707070u) & ~vsc & 0x80808080u) != 0u), 0)) over_step = true;
            }
            uint16_t* vs16 = reinterpret_cast<uint16_t*>(sm + OFF_VS) + lane;
            uint16_t* vz16 = reinterpret_cast<uint16_t*>(sm + OFF_VZ) + lane;
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2) {
                // f16 2^e of two channel groups: (e + 15) << 10 per half; below 2^-15 the step is
                // immaterial and is held there
                const uint32_t e2 = __builtin_amdgcn_perm(0u, vsc, h2 ? 0x030C020Cu : 0x010C000Cu);   // (e << 8) pairs
                constexpr short LEAST = (ANY ? -126 : LONG ? MIN_STEP_EXP : -15) * 256;
                const s16x2 ec = __builtin_elementwise_min(
                    __builtin_elementwise_max(__builtin_bit_cast(s16x2, e2), s16x2{LEAST, LEAST}),
                    s16x2{MAX_STEP_EXP * 256, MAX_STEP_EXP * 256});
                if constexpr (LONG && !ANY) v_out |= e2 ^ __builtin_bit_cast(uint32_t, ec);
                const u16x2 st = __builtin_bit_cast(u16x2, ec) * u16x2{4, 4} + u16x2{0x3C00, 0x3C00};
                uint32_t s2 = __builtin_bit_cast(uint32_t, st);
                if constexpr (ANY)         // (2^-15 to 2^-24 are subnormal f16, smaller steps zero)
                    s2 = pack_f16x2(__uint_as_float(static_cast<uint32_t>((ec[0] >> 8) + 127) << 23),
                                    __uint_as_float(static_cast<uint32_t>((ec[1] >> 8) + 127) << 23));
                vs16[(2 * h2) * PT_ROW] = static_cast<uint16_t>(s2);
                vs16[(2 * h2 + 1) * PT_ROW] = static_cast<uint16_t>(s2 >> 16);
                const uint32_t z2 = pack_f16x2(__uint_as_float(vzp[h2] << 16), __uint_as_float(vzp[h2] & 0xFFFF0000u));
                vz16[(2 * h2) * PT_ROW] = static_cast<uint16_t>(z2);
                vz16[(2 * h2 + 1) * PT_ROW] = static_cast<uint16_t>(z2 >> 16);
            }
        }
        if (more) fetch_v();

        // whether a V vector whose step was held has a code that is not zero (one that does not vary has none)
        auto v_needs_other_form = [&](bool held) {
            const uint32_t* vt = reinterpret_cast<const uint32_t*>(sm + OFF_VT) + lane;
            const uint16_t* vs16 = reinterpret_cast<const uint16_t*>(sm + OFF_VS) + lane;
            bool bad = false;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const uint32_t step = vs16[c * PT_ROW];
                bad |= (step == 0x0400u || step == 0x7800u) && (vt[2 * c * VT_COL] | vt[(2 * c + 1) * VT_COL]) != 0;
            }
            return any_lane(held && bad);
        };

        // ------------------------------------------------------------------ softmax
        if constexpr (NH == 4) {
            // the lane owns token n0 + lane and the four heads; bias of (group, head) = sum q*zp - sum A*2^e
            float x[4];
            {
                const int gsel = lane >> 5;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    // lane 0 / 1 of every row: column 0 / 1 (zp) minus column 2 / 3 (2^e)
                    // (each row goes through a register of its own first: read straight out of the 4-register
                    // result, the four moves came out as one, all reading row 0)
                    float mine = dbias[r];
                    asm volatile("" : "+v"(mine));
                    const float other = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
                        0, __builtin_bit_cast(int, mine), 0x4E, 0xF, 0xF, true));     // quad_perm [2,3,0,1]
                    x[r] = dsel[0][r] + lane_value(mine - other, gsel);
                }
            }
            float pe[4];          // base-2 logit minus the running maximum
            if (a.cap > 0.0f) {
                asm volatile("" ::: "memory");
#pragma unroll
                for (int r = 0; r < 4; ++r) x[r] = apply_cap(x[r] * sm_scale, a.cap) * 1.4426950408889634f;
#pragma unroll
                for (int r = 0; r < 4; ++r) pe[r] = x[r] - m_run[r];
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    x[r] *= c2;
                    pe[r] = x[r] - m_run[r];
                }
            }
            const bool tok_ok = n0 + lane < n_end;
            if (n0 + 64 > n_end) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (!tok_ok) { x[r] = -INFINITY; pe[r] = -INFINITY; }
                }
            }
            // (longer groups: a V step for the other form is seen to here, before it is summed)
            if (any_lane(fmaxf(fmaxf(pe[0], pe[1]), fmaxf(pe[2], pe[3])) > MAX_SLACK<LONG> || (LONG && !ANY && v_out != 0))) {
                if constexpr (LONG && !ANY) {
                    if (__builtin_expect(any_lane(v_out != 0), 0)) {
                        if (v_needs_other_form(v_out != 0)) goto other_form;
                    }
                }
                // refresh the running maxima (always on the first step) and rescale what is summed so far
                float mxs[4] = {x[0], x[1], x[2], x[3]};
                wave_max4(mxs);
                float alpha[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float m_new = fmaxf(m_run[r], mxs[r]);
                    alpha[r] = (m_run[r] == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(m_run[r] - m_new);
                    m_run[r] = m_new;
                    pe[r] = x[r] - m_new;
                }
                // accumulators hold column (x, head j % 4) in every register
                const float al = (j & 3) == 0 ? alpha[0] : ((j & 3) == 1 ? alpha[1] : ((j & 3) == 2 ? alpha[2] : alpha[3]));
#pragma unroll
                for (int i = 0; i < 4; ++i) { acc[0][i] *= al; acc[1][i] *= al; accz[i] *= al; }
            }
            {
                // (to the nearest f16: the pairwise conversion cuts off, which costs half an instruction less a
                // weight and shifts every lse by -2.4e-4 and with it the share of the bf16 tail)
                _Float16* pt = reinterpret_cast<_Float16*>(sm + OFF_PT) + lane;
#pragma unroll
                for (int r = 0; r < 4; ++r) pt[r * PT_ROW] = static_cast<_Float16>(__builtin_amdgcn_exp2f(pe[r]));
            }
        } else {
            // the lane owns tokens n0 + 32g + 16(kq >> 1) + j, g = 0, 1, and heads 4(kq & 1)..+3.  Every quad
            // of a row holds the bias columns (zp g0, zp g1, 2^e g0, 2^e g1) of the row's own heads.
            float x[2][4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float mine = dbias[r];
                asm volatile("" : "+v"(mine));
                const float other = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
                    0, __builtin_bit_cast(int, mine), 0x4E, 0xF, 0xF, true));     // quad_perm [2,3,0,1]
                float t = mine - other;                                           // lanes 0, 1 of a quad: bias of group 0, 1
                asm volatile("" : "+v"(t));
                x[0][r] = dsel[0][r] + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
                    0, __builtin_bit_cast(int, t), 0x00, 0xF, 0xF, true));        // quad_perm [0,0,0,0]
                x[1][r] = dsel[1][r] + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
                    0, __builtin_bit_cast(int, t), 0x55, 0xF, 0xF, true));        // quad_perm [1,1,1,1]
            }
            float pe[2][4];
            if (a.cap > 0.0f) {
                asm volatile("" ::: "memory");
#pragma unroll
                for (int g = 0; g < 2; ++g)
#pragma unroll
                    for (int r = 0; r < 4; ++r) x[g][r] = apply_cap(x[g][r] * sm_scale, a.cap) * 1.4426950408889634f;
            } else {
#pragma unroll
                for (int g = 0; g < 2; ++g)
#pragma unroll
                    for (int r = 0; r < 4; ++r) x[g][r] *= c2;
            }
            const int tk = 16 * (kq >> 1) + j;           // the lane's token inside either group
            if (n0 + 64 > n_end) {
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    const bool tok_ok = n0 + 32 * g + tk < n_end;
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (!tok_ok) x[g][r] = -INFINITY;
                }
            }
            float over = -INFINITY;
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    pe[g][r] = x[g][r] - m_run[r];
                    over = fmaxf(over, pe[g][r]);
                }
            if (any_lane(over > MAX_SLACK<LONG> || (LONG && !ANY && v_out != 0))) {
                if constexpr (LONG && !ANY) {
                    if (__builtin_expect(any_lane(v_out != 0), 0)) {
                        if (v_needs_other_form(v_out != 0)) goto other_form;
                    }
                }
                // refresh the running maxima of the lane's four heads (rows kq and kq ^ 2 hold the same
                // heads) and rescale what is summed so far
                float mxs[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) mxs[r] = fmaxf(x[0][r], x[1][r]);
                rowpair_max4(mxs);
                float alpha[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float m_new = fmaxf(m_run[r], mxs[r]);
                    alpha[r] = (m_run[r] == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(m_run[r] - m_new);
                    m_run[r] = m_new;
                    pe[0][r] = x[0][r] - m_new;
                    pe[1][r] = x[1][r] - m_new;
                }
                // accumulators hold column (x, head j % 8) in every register: the factor of that head is
                // the lane's own when (j >> 2 & 1) == (kq & 1), else that of the neighbouring row
                float al_own = (j & 3) == 0 ? alpha[0] : ((j & 3) == 1 ? alpha[1] : ((j & 3) == 2 ? alpha[2] : alpha[3]));
                const float al_nb = lane_value(al_own, lane ^ 16);
                const float al = (((j >> 2) & 1) == (kq & 1)) ? al_own : al_nb;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    acc[0][i] *= al; acc[1][i] *= al; acc[2][i] *= al; acc[3][i] *= al; accz[i] *= al;
                }
            }
            {
                _Float16* pt = reinterpret_cast<_Float16*>(sm + OFF_PT) + 4 * (kq & 1) * PT_ROW + tk;
#pragma unroll
                for (int g = 0; g < 2; ++g)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        pt[32 * g + r * PT_ROW] = static_cast<_Float16>(__builtin_amdgcn_exp2f(pe[g][r]));
            }
        }
        lds_fence();

        // ------------------------------------------------------------------ P.V (transposed)
        // Lane addresses of this phase, formed here from the lane number rather than carried through
        // the QK phase, where registers are shortest (the copy below keeps them from being hoisted).
        // Row i = j of the V operand is channel 16*(j & 7) + 8*(j >> 3) + Y; column j is (x = j >> 2, head j & 3),
        // or (x = j >> 3, head j & 7) with 8 heads.
        int lane_pv = lane;
        asm volatile("" : "+v"(lane_pv));
        const int jp = lane_pv & 15, kqp = lane_pv >> 4;
        const uint32_t vt_addr = OFF_VT + ((jp & 7) * VT_COL + 8 * kqp) * 4;
        const uint32_t vs_addr = OFF_VS + (((jp & 7) >> 1) * PT_ROW + 8 * kqp) * 2;
        const uint32_t pt_addr = OFF_PT + ((jp & (NH - 1)) * PT_ROW + 8 * kqp) * 2;
        // rows of the sums operand: 0-3 V zero points, 4-7 V steps, 8 ones, others zero
        // (ANY: no constants to take out, so zeros in the place of the steps)
        const uint32_t az_addr = jp < (ANY ? 4 : 8) ? OFF_VZ + (jp * PT_ROW + 8 * kqp) * 2 : (jp == 8 ? OFF_ONES : OFF_ZERO) + 16 * kqp;
        const uint32_t vsel = (jp & 8) ? 0x07060302u : 0x05040100u;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            if (kb == 1 && !g1_live) break;
            // sums: rows vz[cg], 2^e[cg], ones against the weights of column (x, head)
            const u32x4 pw = *reinterpret_cast<const u32x4*>(sm + pt_addr + 64 * kb);
            const u32x4 az = *reinterpret_cast<const u32x4*>(sm + az_addr + 64 * kb);
            accz = mfma_f16(az, pw, accz);
            const u32x4 sw = *reinterpret_cast<const u32x4*>(sm + vs_addr + 64 * kb);
            const u32x4 va = *reinterpret_cast<const u32x4*>(sm + vt_addr + 128 * kb);
            const u32x4 vb = *reinterpret_cast<const u32x4*>(sm + vt_addr + 128 * kb + 16);
            const uint32_t mg0 = __builtin_amdgcn_perm(va[1], va[0], vsel);
            const uint32_t mg1 = __builtin_amdgcn_perm(va[3], va[2], vsel);
            const uint32_t mg2 = __builtin_amdgcn_perm(vb[1], vb[0], vsel);
            const uint32_t mg3 = __builtin_amdgcn_perm(vb[3], vb[2], vsel);
            if constexpr (NH == 4) {
                // column replica x takes the channel blocks Y with Y % 4 == x: for the others the weights are zeroed
#define OMMX_PVX(X)                                                                                       \
                {                                                                                         \
                    const bool mine = (jp >> 2) == X;                                                     \
                    const u32x4 bx = {mine ? pw[0] : 0u, mine ? pw[1] : 0u, mine ? pw[2] : 0u, mine ? pw[3] : 0u}; \
                    acc[0] = mfma_f16(u32x4{v_op<X, LONG, ANY>(mg0, sw[0]), v_op<X, LONG, ANY>(mg1, sw[1]),                 \
                                            v_op<X, LONG, ANY>(mg2, sw[2]), v_op<X, LONG, ANY>(mg3, sw[3])}, bx, acc[0]);   \
                    acc[1] = mfma_f16(u32x4{v_op<4 + X, LONG, ANY>(mg0, sw[0]), v_op<4 + X, LONG, ANY>(mg1, sw[1]),         \
                                            v_op<4 + X, LONG, ANY>(mg2, sw[2]), v_op<4 + X, LONG, ANY>(mg3, sw[3])}, bx, acc[1]); \
                }
                OMMX_PVX(0) OMMX_PVX(1) OMMX_PVX(2) OMMX_PVX(3)
#undef OMMX_PVX
            } else {
                // two column replicas: x takes the channel blocks Y with Y % 2 == x; blocks 2i and 2i + 1 share
                // accumulator i
                const bool first = (jp >> 3) == 0;
                const u32x4 bx0 = {first ? pw[0] : 0u, first ? pw[1] : 0u, first ? pw[2] : 0u, first ? pw[3] : 0u};
                const u32x4 bx1 = {first ? 0u : pw[0], first ? 0u : pw[1], first ? 0u : pw[2], first ? 0u : pw[3]};
#define OMMX_PVY(Y)                                                                                       \
                acc[(Y) >> 1] = mfma_f16(u32x4{v_op<Y, LONG, ANY>(mg0, sw[0]), v_op<Y, LONG, ANY>(mg1, sw[1]),              \
                                               v_op<Y, LONG, ANY>(mg2, sw[2]), v_op<Y, LONG, ANY>(mg3, sw[3])},             \
                                         ((Y) & 1) ? bx1 : bx0, acc[(Y) >> 1]);
                OMMX_PVY(0) OMMX_PVY(1) OMMX_PVY(2) OMMX_PVY(3) OMMX_PVY(4) OMMX_PVY(5) OMMX_PVY(6) OMMX_PVY(7)
#undef OMMX_PVY
            }
        }
        lds_fence();
    }

    report_table_range(a.err, bad_id);
    if (over_step && a.err && lane == 0) atomicOr(a.err, OMMX_ERR_VALUE_RANGE);

    // ---- epilogue: o = (f*(acc - sum p*2^e) + sum p*zp) / l, f = 16 or 4; lse = m + ln l ----------
    // sums live in the lanes of the same column j: rows 0-3 (kq 0) zero points, 4-7 (kq 1) steps, 8 (kq 2) ones
    // (lane-derived values are formed afresh here: carried over from the top of the kernel they
    // would sit in registers the loop needs, or in scratch memory)
    int lane_e = lane;
    asm volatile("" : "+v"(lane_e));
    const int je = lane_e & 15, kqe = lane_e >> 4;
    const int h = je & (NH - 1), x = NH == 8 ? je >> 3 : je >> 2;
    const float l_tot = lane_value(accz[0], 32 + je);
    float z4[4], s4[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        z4[r] = lane_value(accz[r], je);
        s4[r] = lane_value(accz[r], 16 + je);
    }
    const float inv = l_tot > 0.0f ? __builtin_amdgcn_rcpf(l_tot) : 0.0f;
    if (h < heads) {
        float* dst = a.al + b * a.al_b + (int64_t)(qh0 + h) * a.al_h + (int64_t)sp * a.al_s;
#pragma unroll
        for (int a2 = 0; a2 < NH / 2; ++a2) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                // row i = 4kq + r of block Y (4*a2 + x with 4 heads, 2*a2 + x with 8): channel
                // 16*(i & 7) + 8*(i >> 3) + Y, group (i & 7) / 2
                const float pz = (r >> 1) ? ((kqe & 1) ? z4[3] : z4[1]) : ((kqe & 1) ? z4[2] : z4[0]);
                const float psum = (r >> 1) ? ((kqe & 1) ? s4[3] : s4[1]) : ((kqe & 1) ? s4[2] : s4[0]);
                const int ch = 64 * (kqe & 1) + 16 * r + 8 * (kqe >> 1) + (NH == 8 ? 2 : 4) * a2 + x;
                const float f = LONG || (x & 1) ? 4.0f : 16.0f;
                const float val = (f * (acc[a2][r] - psum) + pz) * inv;
                if (!half) dst[ch] = val;
                else if ((kqe & 1) == h / r_half) dst[ch & 63] = val;     // the head's own 64 channels
            }
        }
        // the running maximum of head h: with 8 heads it lives in the rows with (kq & 1) == h >> 2
        if (x == 0 && kqe == (NH == 8 ? (h >> 2) : 0)) {
            const int hr = h & 3;
            const float mt = hr == 0 ? m_run[0] : (hr == 1 ? m_run[1] : (hr == 2 ? m_run[2] : m_run[3]));
            a.sl[b * a.sl_b + (int64_t)(qh0 + h) * a.sl_h + (int64_t)sp * a.sl_s] = l_tot > 0.0f ? (mt + log2f(l_tot)) * 0.6931471805599453f : -INFINITY;
        }
    }
