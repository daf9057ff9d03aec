// Dealing the packed groups of a batch out to workgroups in equal shares.
//
// With a fixed number of splits per request, requests of different length give workgroups of different length: the
// launcher had to start two or four rounds of them to even out (every workgroup pays about one 64-token step of start-up,
// and every split a partial state of 516 bytes per q head that is written and read again).  Here the
// kernel itself cuts the batch into at most `shares` pieces of at most g groups, g the smallest number for
// which every request's ceil(groups / g) pieces fit: one round of workgroups that are all resident and all
// about equally long.  Every wave works this out from the lengths alone (64 lanes, one request each, or four),
// a few hundred instructions that run while the first loads would be waiting for their addresses anyway.
// Measured for the whole call, fixed splits -> shares: 32 requests of 1 to 16 K tokens 108 -> 101 us, 5 of 3.6 to
// 7.6 K at head_dim 64 30.8 -> 25.6, 8 of 3936 with 64 q heads 34.0 -> 28.4, 25 of 1.1 to 5.3 K 54.5 -> 48.7.
#pragma once
#include "ommx_decode_args.h"

namespace ommx {
namespace shares {

// Inclusive sum over the lanes; lane 63 holds the total.
__device__ __forceinline__ uint32_t lane_scan(uint32_t v) {
#define OMMX_DPP_ADD(CTRL, ROWS) v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, ROWS, 0xF, false))
    OMMX_DPP_ADD(0x111, 0xF);        // row_shr:1, 2, 4, 8
    OMMX_DPP_ADD(0x112, 0xF);
    OMMX_DPP_ADD(0x114, 0xF);
    OMMX_DPP_ADD(0x118, 0xF);
    OMMX_DPP_ADD(0x142, 0xA);        // row_bcast:15 into rows 1 and 3
    OMMX_DPP_ADD(0x143, 0xC);        // row_bcast:31 into rows 2 and 3
#undef OMMX_DPP_ADD
    return v;
}
// Maximum over the lanes, uniform.
__device__ __forceinline__ uint32_t lane_max(uint32_t v) {
#define OMMX_DPP_MAX(CTRL, ROWS) v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, ROWS, 0xF, false)))
    OMMX_DPP_MAX(0x111, 0xF);
    OMMX_DPP_MAX(0x112, 0xF);
    OMMX_DPP_MAX(0x114, 0xF);
    OMMX_DPP_MAX(0x118, 0xF);
    OMMX_DPP_MAX(0x142, 0xA);
    OMMX_DPP_MAX(0x143, 0xC);
#undef OMMX_DPP_MAX
    return __builtin_amdgcn_readlane(static_cast<int>(v), 63);
}
__device__ __forceinline__ uint32_t lane_top(uint32_t v) { return __builtin_amdgcn_readlane(static_cast<int>(v), 63); }

struct Share {
    int b, L;            // request and its packed length
    uint32_t sp, n;      // share number sp of the request's n
};

// Clocks a wave spends on g groups (a step is two; a lone group costs 0.7 of one, the start-up about one),
// next to one other wave on its SIMD and next to two: 11 700 and 15 900 a step, here in hundreds.
template <int GT>
__device__ __forceinline__ uint32_t wave_cost(uint32_t g, bool third) {
    return ((GT == 32 ? (g >> 1) * 10u + (g & 1u) * 7u : g * 10u) + 10u) * (third ? 159u : 117u);
}

// The share `f` of the batch; false when the batch has fewer.  GT: tokens per group, PER_LANE: requests per lane
// (B <= 64 * PER_LANE).  The launcher sees to shares >= shares_few >= B, so the search ends at the latest when g is
// the longest request.
// OF_REQUEST: f is a request, of which only L and n are looked up.
// (Args: DecodeArgs, or what else has its fields)
template <int GT, int PER_LANE, bool OF_REQUEST = false, class Args>
__device__ __forceinline__ bool find_share(const Args& a, uint32_t f, int lane, Share& out) {
    int len[PER_LANE];
    uint32_t G[PER_LANE], total = 0, top = 0;
#pragma unroll
    for (int r = 0; r < PER_LANE; ++r) {
        const int idx = 64 * r + lane;
        len[r] = idx < a.B ? a.seq[idx] : 0;
        // (an empty request has one share too: somebody has to write that nothing was attended)
        G[r] = idx < a.B ? max(1u, static_cast<uint32_t>(max(len[r], 0) + GT - 1) / GT) : 0u;
        total += G[r];
        top = max(top, G[r]);
    }
    total = lane_top(lane_scan(total));
    top = lane_max(top);
    const uint32_t most = a.S;
    uint32_t n[PER_LANE], incl[PER_LANE];
    auto deal = [&](uint32_t g) {             // pieces of at most g groups: how many in all
        uint32_t before = 0;
#pragma unroll
        for (int r = 0; r < PER_LANE; ++r) {
            n[r] = g == 1 ? G[r] : (G[r] + g - 1) / g;
            incl[r] = lane_scan(n[r]) + before;
            before = lane_top(incl[r]);
        }
        return before;
    };
    // the smallest g from g0 on whose pieces fit: total / want, and no more than total / (want - B) (each request's last
    // piece may be short) or than the longest request
    auto smallest = [&](uint32_t want, uint32_t g0) {
        uint32_t lo = max(g0, (total + want - 1) / want);
        if (deal(lo) <= want) return lo;
        const uint32_t B = static_cast<uint32_t>(a.B);
        uint32_t hi = max(lo, want > B ? min(top, (total + want - B - 1) / (want - B)) : top);
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (deal(mid) <= want) hi = mid;
            else lo = mid + 1;
        }
        deal(lo);
        return lo;
    };
    // single groups only while waves are short: with the chip full, pairs (one step) walk as fast and leave half the states
    uint32_t g0 = total > static_cast<uint32_t>(a.singles) && GT == 32 ? 2u : 1u;
    if (top > most) g0 = max(g0, (top + most - 1) / most);
    uint32_t g = smallest(a.shares_few, g0);
    if (a.shares > a.shares_few && g > g0) {
        const uint32_t g3 = smallest(a.shares, g0);
        if (wave_cost<GT>(g3, true) < wave_cost<GT>(g, false)) g = g3;
        else deal(g);
    }
    if constexpr (OF_REQUEST) {
        static_assert(PER_LANE == 1, "one request a lane");
        out.b = static_cast<int>(f);
        out.n = __builtin_amdgcn_readlane(static_cast<int>(n[0]), f);
        out.sp = 0;
        out.L = __builtin_amdgcn_readlane(len[0], f);
        return true;
    }
    if (f >= lane_top(incl[PER_LANE - 1])) return false;
#pragma unroll
    for (int r = 0; r < PER_LANE; ++r) {
        const uint64_t hit = __ballot(f < incl[r] && f + n[r] >= incl[r] && n[r] > 0);
        if (hit) {
            const int l = __builtin_ctzll(hit);
            out.b = 64 * r + l;
            out.n = __builtin_amdgcn_readlane(static_cast<int>(n[r]), l);
            out.sp = f + out.n - static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(incl[r]), l));
            out.L = __builtin_amdgcn_readlane(len[r], l);
        }
    }
    // what the combine needs to know about this request
    if (out.sp == 0 && blockIdx.x == 0 && threadIdx.x == 0) a.share_count[out.b] = static_cast<int32_t>(out.n);
    return true;
}

}  // namespace shares
}  // namespace ommx
