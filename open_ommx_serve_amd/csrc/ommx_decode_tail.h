// The bf16 tail rows (sink and recent) of a request attended inside the split-KV launch, as kTailParts more states beside
// the splits' own: a wave takes a quarter of the rows of one kv head.
//
// Attending them in the merge put their whole chain -- length, rows, logits, softmax, P.V -- behind the split-KV kernel,
// where it was most of the merge's time.  Here the last workgroups of that launch do it: on compute units that short
// splits leave free, and in full batches while the last shares run out (their waves end 3 us apart).  The merge
// (fold_kernel) is left with one round of loads: 4.6-5.0 -> 3.0-3.7 us at 1 K, 8.0 -> 3.7 us for 8 short requests over a row
// history, whose length and slot are two more dependent loads.  Whole call: 1 K 12.0 -> 10.5 us, 3 requests of 0.7 to 9 K
// with one kv head 14.6 -> 13.0, 32 of 1 to 16 K 101.6 -> 98.9, 8 of 32 K with 64 q heads 107.5 -> 105.9, 16 of 2 to 16 K
// with 64 q heads 75.8 -> 66.5.  In front of the shares, or only where slots are free, the full batches gain nothing.
// Four waves a kv head: the quarter's rows and its 8 or 16 output channels fit registers, and the slowest wave stays
// below a lone split's 6.4 us.
//
// Precision is that of an fp32 softmax: q.k of bf16 operands on the matrix cores is exact in its products and summed in
// fp32, the weights stay fp32 and P.V runs on the vector ALU.
#pragma once
#include "ommx_decode_util.h"

namespace ommx {
namespace tail {

template <int CTRL>
__device__ __forceinline__ float dpp_of(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
// maximum / sum over each row of 16 lanes, left in every lane of the row
__device__ __forceinline__ float row16_max(float v) {
    v = fmaxf(v, dpp_of<0xB1>(v));       // quad_perm [1,0,3,2]
    v = fmaxf(v, dpp_of<0x4E>(v));       // quad_perm [2,3,0,1]
    v = fmaxf(v, dpp_of<0x141>(v));      // row_half_mirror
    v = fmaxf(v, dpp_of<0x140>(v));      // row_mirror
    return v;
}
__device__ __forceinline__ float row16_sum(float v) {
    v += dpp_of<0xB1>(v);
    v += dpp_of<0x4E>(v);
    v += dpp_of<0x141>(v);
    v += dpp_of<0x140>(v);
    return v;
}
// Sums over the lanes 32 (16) apart of two registers at once: x's in the lower half (even rows), y's in the upper half
// (odd rows).
__device__ __forceinline__ float fold32(float x, float y) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float fold16(float x, float y) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// A store that other workgroups of the same launch may read: it goes past this die's cache.
template <bool SHARED>
__device__ __forceinline__ void put2(float* p, float x, float y) {
    if constexpr (SHARED) {
        const uint64_t v = static_cast<uint64_t>(__float_as_uint(y)) << 32 | __float_as_uint(x);
        __hip_atomic_store(reinterpret_cast<uint64_t*>(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
        *reinterpret_cast<f32x2*>(p) = f32x2{x, y};
    }
}
template <bool SHARED>
__device__ __forceinline__ void put1(float* p, float x) {
    if constexpr (SHARED) __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *p = x;
}

// RT: q head slots (4 or 8; slots from R on repeat the last head and are not written).  LDS: 32 * RT + 2 * RT floats.  SHARED: the states are
// read by another workgroup of this launch.
// (Args: DecodeArgs, or what else has its fields)
template <int RT, int D, bool SHARED = false, class Args>
__device__ __forceinline__ void attend_part(const Args& a, uint8_t* sm, int b, int kvh, int R, int part, int lane) {
    constexpr int CHUNK = 32;                      // rows per pass: two blocks of 16
    constexpr int KS = D / 32;                     // k-steps of a logit
    constexpr int LPR = D / 8;                     // lanes that read a V row
    constexpr int NRG = 64 / LPR, VI = CHUNK / NRG;
    float* const s_p = reinterpret_cast<float*>(sm);               // [CHUNK][RT]
    float* const s_alpha = s_p + CHUNK * RT;                       // [RT]
    float* const s_l = s_alpha + RT;                               // [RT]
    const int j = lane & 15, kq = lane >> 4;
    const int qh0 = kvh * R;
    // one row map for both kinds of tail: gathered rows are row t of the request (no sliding part)
    TailRows<true> rows;
    if (a.t.hist_seq) {
        rows.init(a.t, b);
    } else {
        TailRows<false> plain;
        plain.init(a.t, b);
        rows.n = rows.n_sink = plain.n;
        rows.k_base = plain.k_base;
        rows.v_base = plain.v_base;
        rows.turn = rows.span = rows.sink = 0;
        rows.cap = 1;
    }
    // q of head j % RT: k = (ks, kq, i) <-> channel 32 ks + 8 kq + i
    typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
    u32x4 aq[KS];
    {
        const uint16_t* qp = a.q + (int64_t)b * a.q_sb + (int64_t)(qh0 + min(j & (RT - 1), R - 1)) * a.q_sh + 8 * kq;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) aq[ks] = *reinterpret_cast<const u32x4_a4*>(qp + 32 * ks);
    }
    const int n = rows.n, per = ((n + 15) >> 4) * 4;
    const int lo = part * per, hi = min(n, lo + per);
    float m_run[4], l_run[4], acc[RT][8];
#pragma unroll
    for (int r = 0; r < 4; ++r) { m_run[r] = -INFINITY; l_run[r] = 0.0f; }
#pragma unroll
    for (int h = 0; h < RT; ++h)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[h][e] = 0.0f;
    const int rg = lane / LPR, c8 = lane % LPR;
    for (int r0 = lo; r0 < hi; r0 += CHUNK) {
        // every row of the pass is asked for at once; rows past the part repeat its last one and get no weight
        u32x4 kk[2][KS], vv[VI];
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
            const uint16_t* kp = a.t.kt + rows.k_base + (int64_t)rows.row(min(r0 + 16 * tb + j, hi - 1)) * a.t.kt_t +
                                 (int64_t)kvh * a.t.kt_h + 8 * kq;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) kk[tb][ks] = *reinterpret_cast<const u32x4*>(kp + 32 * ks);
        }
#pragma unroll
        for (int i = 0; i < VI; ++i)
            vv[i] = *reinterpret_cast<const u32x4*>(a.t.vt + rows.v_base + (int64_t)rows.row(min(r0 + rg + NRG * i, hi - 1)) * a.t.vt_t +
                                                    (int64_t)kvh * a.t.vt_h + 8 * c8);
        f32x4 d[2] = {f32x4{0, 0, 0, 0}, f32x4{0, 0, 0, 0}};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) d[tb] = decode_util::mfma_bf16(aq[ks], kk[tb][ks], d[tb]);
        // result row 4 kq + r is head (4 kq + r) % RT, column j the token
        float p[2][4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float x[2];
#pragma unroll
            for (int tb = 0; tb < 2; ++tb)
                x[tb] = r0 + 16 * tb + j < hi ? apply_cap(d[tb][r] * a.sm_scale, a.cap) : -INFINITY;
            const float m_new = fmaxf(m_run[r], row16_max(fmaxf(x[0], x[1])));
            const float m_safe = m_new == -INFINITY ? 0.0f : m_new;        // (a row of infinite logits)
            const float alpha = m_run[r] == -INFINITY ? 0.0f : __expf(m_run[r] - m_safe);
            m_run[r] = m_new;
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) p[tb][r] = x[tb] == -INFINITY ? 0.0f : __expf(x[tb] - m_safe);
            l_run[r] = l_run[r] * alpha + (p[0][r] + p[1][r]);
            if (r0 > lo && j == 0 && kq < RT / 4) s_alpha[4 * kq + r] = alpha;
        }
        decode_util::lds_fence();
        {
            const int tb = RT == 4 ? kq : kq >> 1;          // (the replicas of a result each write one block of it)
            const f32x4 mine = tb == 0 ? f32x4{p[0][0], p[0][1], p[0][2], p[0][3]} : f32x4{p[1][0], p[1][1], p[1][2], p[1][3]};
            if (tb < 2) *reinterpret_cast<f32x4*>(s_p + (16 * tb + j) * RT + (RT == 4 ? 0 : 4 * (kq & 1))) = mine;
        }
        decode_util::lds_fence();
        if (r0 > lo) {
#pragma unroll
            for (int h = 0; h < RT; ++h) {
                const float al = s_alpha[h];
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[h][e] *= al;
            }
        }
#pragma unroll
        for (int i = 0; i < VI; ++i) {
            const int t = rg + NRG * i;
            float v[8];
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                v[2 * w] = __uint_as_float(vv[i][w] << 16);
                v[2 * w + 1] = __uint_as_float(vv[i][w] & 0xFFFF0000u);
            }
            // (rows past the part: weight zero times a row that is there; an infinite row must not become NaN by that)
            if (r0 + t < hi) {
#pragma unroll
                for (int h4 = 0; h4 < RT / 4; ++h4) {
                    const f32x4 w4 = *reinterpret_cast<const f32x4*>(s_p + t * RT + 4 * h4);
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int e = 0; e < 8; ++e) acc[4 * h4 + r][e] = fmaf(w4[r], v[e], acc[4 * h4 + r][e]);
                }
            }
        }
        decode_util::lds_fence();
    }
    // ---- the state: sums over the lanes, normalised ----------------------------------------------
    float* const al = a.al + (int64_t)b * a.al_b + (int64_t)qh0 * a.al_h + (int64_t)(part - kTailParts) * a.al_s;
    float* const sl = a.sl + (int64_t)b * a.sl_b + (int64_t)qh0 * a.sl_h + (int64_t)(part - kTailParts) * a.sl_s;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float l = row16_sum(l_run[r]);
        const int h = 4 * kq + r;
        if (j == 0 && kq < RT / 4) {
            s_l[h] = l;
            if (h < R) put1<SHARED>(sl + h * a.sl_h, l > 0.0f ? m_run[r] + __logf(l) : -INFINITY);
        }
    }
    if (lo >= hi) return;                           // (nothing attended: the lse says so, the state is not read)
    decode_util::lds_fence();
#pragma unroll
    for (int h4 = 0; h4 < RT / 4; ++h4) {
        // four heads of eight channels: 32 sums become 8 registers, row kq of lanes holding head 4 h4 + kq
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float even = fold32(acc[4 * h4][e], acc[4 * h4 + 2][e]), odd = fold32(acc[4 * h4 + 1][e], acc[4 * h4 + 3][e]);
            o[e] = fold16(even, odd);
            if (D == 64) o[e] += dpp_of<0x128>(o[e]);          // row_ror:8, the two halves of a row of lanes
        }
        const int h = 4 * h4 + kq;
        if (h < R && (D == 128 || (lane & 8) == 0)) {
            const float inv = 1.0f / s_l[h];
            float* dst = al + h * a.al_h + 8 * c8;
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] *= inv;
            if constexpr (SHARED) {
#pragma unroll
                for (int e = 0; e < 8; e += 2) put2<true>(dst + e, o[e], o[e + 1]);
            } else {
                *reinterpret_cast<f32x4*>(dst) = f32x4{o[0], o[1], o[2], o[3]};
                *reinterpret_cast<f32x4*>(dst + 4) = f32x4{o[4], o[5], o[6], o[7]};
            }
        }
    }
}

}  // namespace tail
}  // namespace ommx
