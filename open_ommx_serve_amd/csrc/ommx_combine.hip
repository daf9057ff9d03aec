// Split combine with the bf16 sink/recent tail folded in.  Follows
// ommx_gpu_serve/attention/paged_decode.py:2366-2500: valid splits are recomputed from the
// packed length with the stage-1 rounding; the tail is one more softmax part computed here from
// k_tail/v_tail; o = sum w_i o_i / sum w_i, lse = max + ln sum w_i; nothing attended gives
// o = 0, lse = -inf.
//
// fold_kernel (at the end) merges when the split-KV launch has attended the tail already; two kernels attend it themselves.
// combine_kernel: Q workgroups per (request, q head), one per piece of the head's
// channels.  It is latency bound (few small workgroups, a few KB each), so every global load is
// issued before the first wait: thread (d, sg) owns channel d of the splits sg, sg+NSG, ... and
// of the tail rows sg, sg+NSG, ...; for the tail logits the same threads regroup as (row, 16
// parts of the row).  combine_grouped_kernel (further down): one workgroup per (request, kv head)
// for large batches, where the tail rows are most of the bytes and are read once for all the
// q heads of the kv head.
#include <algorithm>

#include "ommx_decode_args.h"

namespace ommx {

namespace {
// Lane exchanges inside the vector ALU (DPP): no trip through the LDS crossbar, no index arithmetic.
template <int CTRL>
__device__ __forceinline__ float dpp_of(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
        __builtin_bit_cast(int, v), __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
// sum over each row of 16 lanes, left in every lane of the row
__device__ __forceinline__ float row16_sum(float v) {
    v += dpp_of<0xB1>(v);        // quad_perm [1,0,3,2]
    v += dpp_of<0x4E>(v);        // quad_perm [2,3,0,1]
    v += dpp_of<0x141>(v);       // row_half_mirror
    v += dpp_of<0x140>(v);       // row_mirror
    return v;
}
// maximum over the 64 lanes, uniform
__device__ __forceinline__ float wave64_max(float v) {
    v = fmaxf(v, dpp_of<0xB1>(v));
    v = fmaxf(v, dpp_of<0x4E>(v));
    v = fmaxf(v, dpp_of<0x141>(v));
    v = fmaxf(v, dpp_of<0x140>(v));
    v = fmaxf(v, dpp_of<0x142>(v));      // row_bcast15: lane 15 of a row into the next row
    v = fmaxf(v, dpp_of<0x143>(v));      // row_bcast31: lane 31 into rows 2 and 3
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
}  // namespace

// NT threads per workgroup, at most MAXS splits: 1024 / 256 in general, 512 / 64 when many
// (request, head) pairs with few splits each fill the chip (fewer idle lanes per workgroup).
__device__ __forceinline__ void put_out(const CombineArgs& a, int64_t at, float v) {
    if (a.o16) a.o16[at] = f32_to_bf16_any(v);
    else a.o[at] = v;
}

// HIST: the tail rows lie in a row history instead of a gathered buffer.  SHARED: the number of states is the
// request's own.
template <int D, int Q, bool HIST, bool SHARED, int NT = 1024, int MAXS = 256>
__global__ void __launch_bounds__(NT) combine_kernel(CombineArgs a) {
    constexpr int CH = D / Q;            // channels of this workgroup (one of Q pieces of the head)
    constexpr int NSG = NT / CH;         // split groups: thread (d, sg) owns splits sg, sg + NSG, ...
    static_assert(MAXS <= NT && MAXS % 64 == 0, "one thread per split slot");
    constexpr int NSP = MAXS / NSG;      // split partials per thread, upper bound
    constexpr int ROWS = NT / 16;        // tail rows handled per chunk (64)
    constexpr int PER = ROWS / NSG;      // tail rows per thread in the P.V step
    static_assert(PER >= 1 && NSP % 4 == 0, "thread layout");
    __shared__ float s_q[D];
    __shared__ __attribute__((aligned(16))) float s_logit[ROWS];
    __shared__ float s_acc[NSG][CH];     // per-sg sums of the split part
    __shared__ float s_tacc[NSG][CH];    // per-sg sums of the tail part
    __shared__ float s_w[NSG], s_tl[NSG], s_wmax[MAXS / 64];
    __shared__ __attribute__((aligned(16))) float s_wT[NSG][NSP];   // weight of split sg + NSG*i at [sg][i]
    const int b = blockIdx.x, h = blockIdx.y, cq = blockIdx.z, tid = threadIdx.x;
    const int dl = tid % CH, sg = tid / CH;
    const int d = cq * CH + dl;          // this thread's channel of the head
    const int kvh = h / (a.Hq / a.Hkv);
    const float* base = a.al + b * a.al_b + (int64_t)h * a.al_h;
    // what everything after the split loads waits for: requested first
    TailRows<HIST> rows;
    rows.init(a, b);
    const int tail = rows.n;

    // ---- all loads of the split part --------------------------------------------------
    // They depend on the arguments only, so they go out before anything is read from
    // memory; one pointer per thread, advanced by NSG split slots per load.  (A uniform trip
    // count and a clamped last address keep the loads free of per-lane branches, so they
    // are all in flight together.)
    // With shares the number of states is itself read from memory, one memory latency (0.7 us) later than everything
    // else: what an even deal gives every request goes out before it is here (the slots exist; what an unused one
    // holds is dropped below), the states beyond that once the weights are there.
    float pv[NSP];
    const int n_i = (a.sure + NSG - 1) / NSG;
    {
        const float* p = base + (int64_t)sg * a.al_s + d;
        const int64_t step = NSG * a.al_s;
#pragma unroll
        for (int i = 0; i < NSP; ++i) {
            pv[i] = 0.0f;
            if (i < n_i) {
                const bool inside = sg + NSG * i < a.S;        // only the last trip can fall outside
                pv[i] = *(inside ? p : base + (int64_t)(a.S - 1) * a.al_s + d);
                p += step;
            }
        }
    }
    // Every split wrote its state, an empty one with lse = -inf (paged_decode.py:2262-2284), so the
    // weights follow from the lse column alone, whatever rule dealt the tokens out to the splits
    // (the reference recomputes its rounding here, paged_decode.py:2407-2410).
    float my_lse = -INFINITY;
    if (tid < MAXS && tid < a.S) my_lse = a.sl[b * a.sl_b + (int64_t)h * a.sl_h + (int64_t)tid * a.sl_s];
    const uint32_t q_raw = (a.q && tid < D) ? a.q[b * a.q_sb + (int64_t)h * a.q_sh + tid] : 0u;
    const int S = SHARED ? min(max(a.share_count[b], 1), a.S) : a.S;
    if (SHARED && tid >= S) my_lse = -INFINITY;

    if (tid < D) s_q[tid] = __uint_as_float(q_raw << 16);
    if (tid < MAXS) {
        const float wm = wave64_max(my_lse);
        if ((tid & 63) == 0) s_wmax[tid >> 6] = wm;
    }

    // ---- tail: chunks of ROWS rows (one chunk in practice: sink + recent <= 72 rows) ----
    // Every quarter computes all the logits (they need the whole q and K rows) and its own
    // channels of P.V.
    float t_m = -INFINITY, t_l = 0.0f, t_acc = 0.0f;
    const int row = tid >> 4, part = tid & 15;
    // loads of one chunk: 16 bytes of one K row, PER elements of V; rows from `last` on repeat it
    uint4 ku;
    uint32_t vv[PER];
    auto load_rows = [&](int r0, int last) {
        ku = *reinterpret_cast<const uint4*>(
            a.kt + rows.k_base + (int64_t)rows.row(r0 + min(row, last)) * a.kt_t + (int64_t)kvh * a.kt_h +
            (part * 8) % D);
#pragma unroll
        for (int i = 0; i < PER; ++i)
            vv[i] = a.vt[rows.v_base + (int64_t)rows.row(r0 + min(sg + NSG * i, last)) * a.vt_t +
                         (int64_t)kvh * a.vt_h + d];
    };
    // When the caller has said how many rows the tail buffers hold, the first chunk is asked for
    // here, with the split loads and before the tail length has arrived (its uses below wait for
    // it): rows past the tail are addressable, and neither their logits nor their V are used.
    const bool early = a.T > 0 && (HIST || a.tail != nullptr);
    if (early) load_rows(0, min(ROWS, a.T) - 1);
    for (int r0 = 0; r0 < tail; r0 += ROWS) {
        const int nr = min(ROWS, tail - r0);
        if (!(early && r0 == 0)) load_rows(r0, nr - 1);
        __syncthreads();                              // s_q ready (and previous chunk consumed)
        float dot = 0.0f;
        if (part * 8 < D) {
            const uint32_t w[4] = {ku.x, ku.y, ku.z, ku.w};
            const float* qq = s_q + part * 8;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                dot = fmaf(qq[2 * i], __uint_as_float(w[i] << 16), dot);
                dot = fmaf(qq[2 * i + 1], __uint_as_float(w[i] & 0xFFFF0000u), dot);
            }
        }
        dot = row16_sum(dot);
        if (part == 0) s_logit[row] = row < nr ? apply_cap(dot * a.sm_scale, a.cap) : -INFINITY;
        __syncthreads();
        // maximum of the chunk's logits: one logit per lane, reduced over the wave (every thread
        // reading all ROWS of them cost 16 LDS reads of 16 bytes each); s_logit holds -inf past nr
        static_assert(ROWS <= 64, "one logit per lane");
        const float mx = wave64_max((tid & 63) < ROWS ? s_logit[tid & 63] : -INFINITY);
        const float m_new = fmaxf(t_m, mx);
        const float alpha = (t_m == -INFINITY) ? 0.0f : __expf(t_m - m_new);
        t_l *= alpha;
        t_acc *= alpha;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int r = sg + NSG * i;
            if (r < nr) {
                const float p = __expf(s_logit[r] - m_new);
                t_l += p;
                t_acc = fmaf(p, __uint_as_float(vv[i] << 16), t_acc);
            }
        }
        t_m = m_new;
    }
    __syncthreads();                                  // s_wmax ready

    // ---- split part: weights from the lse column -----------------------------------------
    // One thread per split turns its lse into a weight; the weights are laid out so that
    // thread (d, sg) reads the ones of its splits sg, sg+NSG, ... as float4.
    float g_max = s_wmax[0];
#pragma unroll
    for (int w = 1; w < MAXS / 64; ++w) g_max = fmaxf(g_max, s_wmax[w]);
    const float g_safe = (g_max == -INFINITY) ? 0.0f : g_max;
    if (tid < MAXS) s_wT[tid % NSG][tid / NSG] = my_lse == -INFINITY ? 0.0f : __expf(my_lse - g_safe);
    __syncthreads();
    float acc = 0.0f, wsum = 0.0f;
#pragma unroll
    for (int i4 = 0; i4 < NSP / 4; ++i4) {
        const float4 w4 = reinterpret_cast<const float4*>(s_wT[sg])[i4];
        const float w[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {          // absent splits have weight zero; their slot
            wsum += w[k];                      // may hold anything, so it is not multiplied
            acc = w[k] > 0.0f ? fmaf(w[k], pv[4 * i4 + k], acc) : acc;
        }
    }
    if (SHARED) {
        for (int i = n_i; i * NSG < S; i += 4) {
            float v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = base[(int64_t)min(sg + NSG * (i + u), S - 1) * a.al_s + d];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float w = i + u < NSP ? s_wT[sg][i + u] : 0.0f;
                acc = w > 0.0f ? fmaf(w, v[u], acc) : acc;
            }
        }
    }
    s_acc[sg][dl] = acc;
    s_tacc[sg][dl] = t_acc;
    if (dl == 0) { s_w[sg] = wsum; s_tl[sg] = t_l; }
    __syncthreads();
    if (sg == 0) {
        float A = 0.0f, W = 0.0f, TA = 0.0f, TL = 0.0f;
#pragma unroll
        for (int k = 0; k < NSG; ++k) { A += s_acc[k][dl]; W += s_w[k]; TA += s_tacc[k][dl]; TL += s_tl[k]; }
        const float tail_lse = TL > 0.0f ? t_m + __logf(TL) : -INFINITY;
        const float n_max = fmaxf(g_max, tail_lse);
        const float n_safe = (n_max == -INFINITY) ? 0.0f : n_max;
        const float rs = (g_max == -INFINITY) ? 0.0f : __expf(g_max - n_safe);
        W *= rs;
        A *= rs;
        if (TL > 0.0f) {
            const float w = __expf(tail_lse - n_safe);
            W += w;
            A = fmaf(w, TA / TL, A);
        }
        put_out(a, b * a.o_b + (int64_t)h * a.o_h + d, W > 0.0f ? A / W : 0.0f);
        if (d == 0) a.lse[b * a.lse_b + h] = W > 0.0f ? n_max + __logf(W) : -INFINITY;
    }
}

__device__ __forceinline__ float wave_max_f32(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}
__device__ __forceinline__ float wave_sum_f32(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// The same merge for a whole kv head at a time: one workgroup of 512 threads per (request, kv
// head) serves the R = 4 or 8 q heads of that kv head, so the bf16 tail rows -- most of the bytes
// when there are few splits -- are read once instead of once per q head.  Used when (request, kv
// head) pairs alone fill the chip twice over (then nothing is gained by one workgroup per q
// head) and there are at most 64 splits.  Wave r < R owns the scalars of head r (split weights, running tail maximum
// and sum); the channel work is dealt out as (head, channel) for the splits and as (channel
// pair, row group) for the tail's P.V.
// EARLY: the tail rows of the first pass are asked for before the split part and held in registers
// (32 more: one workgroup per compute unit instead of two, which pays while the grid is no larger
// than the chip).
template <int D, int R, bool EARLY, bool HIST, bool SHARED>
__global__ void __launch_bounds__(512) combine_grouped_kernel(CombineArgs a) {
    constexpr int NT = 512, MAXS = 64;
    constexpr int ROWS = 128;              // tail rows per pass (two per thread of the logit layout)
    constexpr int CHP = D / 8;             // channels per thread of a K row (8 threads per row)
    constexpr int NRG = NT / (D / 2);      // row groups of the P.V layout
    constexpr int HD = (R * D + NT - 1) / NT;   // (head, channel) items per thread
    __shared__ __attribute__((aligned(16))) float s_q[R][D];
    __shared__ float s_w[R][MAXS];
    __shared__ float s_gmax[R], s_W[R], s_alpha[R], s_tm[R], s_tl[R];
    __shared__ float s_logit[R][ROWS];
    __shared__ float s_p[R][ROWS];
    __shared__ float s_red[NRG][R][D];
    const int b = blockIdx.x, kvh = blockIdx.y, tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int h0 = kvh * R;
    const float* base = a.al + b * a.al_b + (int64_t)h0 * a.al_h;
    // (the states of this request: its own number when the work was dealt out in shares)
    const int S = SHARED ? min(max(a.share_count[b], 1), a.S) : a.S;
    TailRows<HIST> rows;
    rows.init(a, b);
    const int tail = rows.n;

    // ---- split weights: wave r, lane s ----------------------------------------------------
    if (a.q) {
        for (int i = tid; i < R * D / 2; i += NT) {
            const int r = i / (D / 2), c2 = i % (D / 2);
            const uint32_t w = *reinterpret_cast<const uint32_t*>(
                a.q + b * a.q_sb + (int64_t)(h0 + r) * a.q_sh + 2 * c2);
            s_q[r][2 * c2] = __uint_as_float(w << 16);
            s_q[r][2 * c2 + 1] = __uint_as_float(w & 0xFFFF0000u);
        }
    }
    if (wave < R) {
        float my_lse = lane < a.S ? a.sl[b * a.sl_b + (int64_t)(h0 + wave) * a.sl_h + (int64_t)lane * a.sl_s] : -INFINITY;
        if (lane >= S) my_lse = -INFINITY;    // an empty split's lse is -inf, an unused slot holds anything
        const float g_max = wave_max_f32(my_lse);
        const float g_safe = (g_max == -INFINITY) ? 0.0f : g_max;
        const float w = my_lse == -INFINITY ? 0.0f : __expf(my_lse - g_safe);
        const float W = wave_sum_f32(w);
        s_w[wave][lane] = w;
        if (lane == 0) { s_gmax[wave] = g_max; s_W[wave] = W; }
    }
    __syncthreads();

    // ---- the tail rows of the first pass are asked for here, before the split part waits for its
    // own loads: thread (row, part) holds CHP channels of K rows row and row + 64, thread (channel
    // pair, row group) the V dwords of rows rg, rg + NRG, ...
    constexpr int VPT = ROWS / NRG;        // V rows per thread and pass
    const int dp = tid % (D / 2), rg = tid / (D / 2);
    uint4 kk[2][CHP / 8];
    uint32_t vv[VPT];
    auto ask_rows = [&](int r0, int nr) {
        const int part = tid & 7, row = tid >> 3;
#pragma unroll
        for (int h2 = 0; h2 < 2; ++h2) {
            const int t = row + 64 * h2;
#pragma unroll
            for (int c8 = 0; c8 < CHP / 8; ++c8) kk[h2][c8] = uint4{0u, 0u, 0u, 0u};
            if (t < nr) {
                const uint16_t* kp = a.kt + rows.k_base + (int64_t)rows.row(r0 + t) * a.kt_t +
                                     (int64_t)kvh * a.kt_h + part * CHP;
#pragma unroll
                for (int c8 = 0; c8 < CHP / 8; ++c8) kk[h2][c8] = reinterpret_cast<const uint4*>(kp)[c8];
            }
        }
        if constexpr (EARLY) {
#pragma unroll
            for (int i = 0; i < VPT; ++i) {
                const int t = rg + NRG * i;
                vv[i] = 0u;
                if (t < nr)
                    vv[i] = *reinterpret_cast<const uint32_t*>(
                        a.vt + rows.v_base + (int64_t)rows.row(r0 + t) * a.vt_t + (int64_t)kvh * a.vt_h + 2 * dp);
            }
        }
    };
    if constexpr (EARLY) ask_rows(0, min(ROWS, tail));

    // ---- split part: item (head, channel) ---------------------------------------------------
    // Every split slot is read (it exists; an absent split's content is stale and is dropped by
    // the select), so that the loads carry no branch and go out eight at a time.
    float A[HD];
#pragma unroll
    for (int k = 0; k < HD; ++k) {
        A[k] = 0.0f;
        const int i = tid + k * NT;
        if (i < R * D) {
            const int r = i / D, d = i % D;
            const float* p = base + (int64_t)r * a.al_h + d;
            float acc = 0.0f;
            for (int s0 = 0; s0 < S; s0 += 8) {
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = p[(int64_t)min(s0 + u, S - 1) * a.al_s];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const float w = s0 + u < S ? s_w[r][s0 + u] : 0.0f;
                    acc = w > 0.0f ? fmaf(w, v[u], acc) : acc;
                }
            }
            A[k] = acc;
        }
    }

    // ---- tail: passes of up to ROWS rows, online over passes ------------------------------
    float m_run = -INFINITY, l_run = 0.0f;          // of head `wave` (waves < R)
    float acc[R][2];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r][0] = acc[r][1] = 0.0f;
    for (int r0 = 0; r0 < tail; r0 += ROWS) {
        const int nr = min(ROWS, tail - r0);
        if (!EARLY || r0 > 0) ask_rows(r0, nr);
        {   // logits: thread (row, part) takes CHP channels of rows row and row + 64
            const int part = tid & 7, row = tid >> 3;
#pragma unroll
            for (int rr = 0; rr < ROWS; rr += 64) {
                const int t = row + rr;
                float dot[R];
#pragma unroll
                for (int r = 0; r < R; ++r) dot[r] = 0.0f;
                if (t < nr) {
#pragma unroll
                    for (int c8 = 0; c8 < CHP / 8; ++c8) {
                        const uint4 ku = kk[rr / 64][c8];
                        const uint32_t w[4] = {ku.x, ku.y, ku.z, ku.w};
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float k0 = __uint_as_float(w[i] << 16);
                            const float k1 = __uint_as_float(w[i] & 0xFFFF0000u);
                            const int c = part * CHP + 8 * c8 + 2 * i;
#pragma unroll
                            for (int r = 0; r < R; ++r)
                                dot[r] = fmaf(s_q[r][c + 1], k1, fmaf(s_q[r][c], k0, dot[r]));
                        }
                    }
                }
#pragma unroll
                for (int r = 0; r < R; ++r) {
#pragma unroll
                    for (int o = 1; o < 8; o <<= 1) dot[r] += __shfl_xor(dot[r], o);
                }
                if (part == 0) {
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        s_logit[r][t] = t < nr ? apply_cap(dot[r] * a.sm_scale, a.cap) : -INFINITY;
                }
            }
        }
        __syncthreads();
        if (wave < R) {   // softmax bookkeeping of head `wave`: rows lane and lane + 64
            const float x0 = s_logit[wave][lane], x1 = s_logit[wave][lane + 64];
            const float m_new = fmaxf(m_run, wave_max_f32(fmaxf(x0, x1)));
            const float alpha = (m_run == -INFINITY) ? 0.0f : __expf(m_run - m_new);
            const float p0 = x0 == -INFINITY ? 0.0f : __expf(x0 - m_new);
            const float p1 = x1 == -INFINITY ? 0.0f : __expf(x1 - m_new);
            l_run = l_run * alpha + wave_sum_f32(p0 + p1);
            m_run = m_new;
            s_p[wave][lane] = p0;
            s_p[wave][lane + 64] = p1;
            if (lane == 0) s_alpha[wave] = alpha;
        }
        __syncthreads();
        {   // P.V: thread (channel pair, row group)
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const float al = s_alpha[r];
                acc[r][0] *= al;
                acc[r][1] *= al;
            }
            if constexpr (EARLY) {
#pragma unroll
                for (int i = 0; i < VPT; ++i) {
                    const int t = rg + NRG * i;
                    if (t < nr) {
                        const float v0 = __uint_as_float(vv[i] << 16), v1 = __uint_as_float(vv[i] & 0xFFFF0000u);
#pragma unroll
                        for (int r = 0; r < R; ++r) {
                            const float p = s_p[r][t];
                            acc[r][0] = fmaf(p, v0, acc[r][0]);
                            acc[r][1] = fmaf(p, v1, acc[r][1]);
                        }
                    }
                }
            } else {
                for (int t = rg; t < nr; t += NRG) {
                    const uint32_t vw = *reinterpret_cast<const uint32_t*>(
                        a.vt + rows.v_base + (int64_t)rows.row(r0 + t) * a.vt_t + (int64_t)kvh * a.vt_h + 2 * dp);
                    const float v0 = __uint_as_float(vw << 16), v1 = __uint_as_float(vw & 0xFFFF0000u);
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const float p = s_p[r][t];
                        acc[r][0] = fmaf(p, v0, acc[r][0]);
                        acc[r][1] = fmaf(p, v1, acc[r][1]);
                    }
                }
            }
        }
        // (the next pass writes s_logit before its first barrier and s_p after it: both are
        // past every read of this pass)
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        s_red[rg][r][2 * dp] = acc[r][0];
        s_red[rg][r][2 * dp + 1] = acc[r][1];
    }
    if (wave < R && lane == 0) { s_tm[wave] = m_run; s_tl[wave] = l_run; }
    __syncthreads();

    // ---- both parts together, item (head, channel) ------------------------------------------
#pragma unroll
    for (int k = 0; k < HD; ++k) {
        const int i = tid + k * NT;
        if (i < R * D) {
            const int r = i / D, d = i % D;
            float TA = 0.0f;
#pragma unroll
            for (int g = 0; g < NRG; ++g) TA += s_red[g][r][d];
            const float TL = s_tl[r], t_m = s_tm[r], g_max = s_gmax[r];
            float W = s_W[r], Av = A[k];
            const float tail_lse = TL > 0.0f ? t_m + __logf(TL) : -INFINITY;
            const float n_max = fmaxf(g_max, tail_lse);
            const float n_safe = (n_max == -INFINITY) ? 0.0f : n_max;
            const float rs = (g_max == -INFINITY) ? 0.0f : __expf(g_max - n_safe);
            W *= rs;
            Av *= rs;
            if (TL > 0.0f) {
                const float w = __expf(tail_lse - n_safe);
                W += w;
                Av = fmaf(w, TA / TL, Av);
            }
            put_out(a, b * a.o_b + (int64_t)(h0 + r) * a.o_h + d, W > 0.0f ? Av / W : 0.0f);
            if (d == 0) a.lse[b * a.lse_b + h0 + r] = W > 0.0f ? n_max + __logf(W) : -INFINITY;
        }
    }
}

// The merge when the tail rows are among the states (ommx_decode_tail.h): o = sum w_i o_i / sum w_i over `slots` states
// of every (request, q head), w_i = exp(lse_i - max).  A workgroup takes CH channels of one head, LPR lanes a state
// (four channels each); every wave reads all the lse and works the maximum and the sum of weights out for itself, so
// that between the one round of loads and the output lie one exchange through LDS and no other wait.  Latency bound, or
// with many heads by how many of them are under way: 32-bit offsets and 47 registers let eight waves a SIMD (as 64-bit
// addresses it took 120 to 130: 48 requests of 64 q heads 80.5 us in all instead of 85, one of 1 K 9.6 instead of 10.2).
// An unused slot has lse -inf, and what it holds is not multiplied.
struct FoldArgs {
    const float* al; int64_t al_b, al_h, al_s;
    const float* sl; int64_t sl_b, sl_h, sl_s;
    float* o; uint16_t* o16; int64_t o_b, o_h;
    float* lse; int64_t lse_b;
    int slots, sure;
};
template <int D, int Q, int NT>
__global__ void __launch_bounds__(NT, 8) fold_kernel(FoldArgs a) {
    constexpr int CH = D / Q, LPR = CH / 4, ROWS = NT / LPR, NW = NT / 64;
    constexpr int FIRST = 6;                       // states per thread of the first round of loads, upper bound
    constexpr int NL = 9;                          // 512 splits and the tail's parts, 64 a register
    static_assert(LPR == 8 || LPR == 16 || LPR == 32, "lane layout of the sums");
    __shared__ float s_acc[NW][CH];
    const int b = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c4 = tid % LPR, row = tid / LPR;
    // (uniform bases, 32-bit offsets behind them: a head's states span less than a megabyte)
    const char* const base = reinterpret_cast<const char*>(a.al + b * a.al_b + (int64_t)h * a.al_h + blockIdx.z * CH);
    const char* const sl = reinterpret_cast<const char*>(a.sl + b * a.sl_b + (int64_t)h * a.sl_h);
    const uint32_t al_s = static_cast<uint32_t>(a.al_s) * 4u, sl_s = static_cast<uint32_t>(a.sl_s) * 4u;
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    auto state = [&](int s) { return *reinterpret_cast<const f32x4*>(base + (static_cast<uint32_t>(s) * al_s + 16u * c4)); };
    auto lse_of = [&](int s) { return *reinterpret_cast<const float*>(sl + static_cast<uint32_t>(s) * sl_s); };
    const int N = a.slots;
    const int n_first = min((a.sure + ROWS - 1) / ROWS, FIRST);
    f32x4 v[FIRST];
    float my[FIRST], all[NL];
#pragma unroll
    for (int i = 0; i < FIRST; ++i) {
        v[i] = f32x4{0, 0, 0, 0};
        my[i] = -INFINITY;
        if (i < n_first) {
            const int s = min(row + ROWS * i, N - 1);
            v[i] = state(s);
            my[i] = lse_of(s);
        }
    }
    float top = -INFINITY;
    int used = 0;                                  // slots up to the last one that holds something
#pragma unroll
    for (int k = 0; k < NL; ++k) {
        all[k] = -INFINITY;
        if (64 * k < N) all[k] = lse_of(min(64 * k + lane, N - 1));
    }
#pragma unroll
    for (int k = 0; k < NL; ++k) {
        if (64 * k < N) {
            if (64 * k + lane >= N) all[k] = -INFINITY;
            const uint64_t live = __ballot(all[k] != -INFINITY);
            if (live) used = 64 * k + 64 - __builtin_clzll(live);
        }
        top = fmaxf(top, all[k]);
    }
    top = wave64_max(top);
    const float safe = top == -INFINITY ? 0.0f : top;
    f32x4 acc = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < FIRST; ++i) {
        if (i < n_first) {
            const float w = my[i] == -INFINITY || row + ROWS * i >= N ? 0.0f : __expf(my[i] - safe);
            if (w > 0.0f) acc += w * v[i];
        }
    }
    for (int s0 = row + ROWS * n_first; s0 < used; s0 += 4 * ROWS) {
        float w[4];
        f32x4 x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) w[u] = lse_of(min(s0 + ROWS * u, used - 1));
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = state(min(s0 + ROWS * u, used - 1));
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            w[u] = w[u] == -INFINITY || s0 + ROWS * u >= used ? 0.0f : __expf(w[u] - safe);
            if (w[u] > 0.0f) acc += w[u] * x[u];
        }
    }
    float W = 0.0f;
#pragma unroll
    for (int k = 0; k < NL; ++k)
        if (64 * k < N) W += all[k] == -INFINITY ? 0.0f : __expf(all[k] - safe);
    W = row16_sum(W);
    {
        auto at = [&](int l) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, W), l)); };
        W = (at(0) + at(16)) + (at(32) + at(48));
    }
    auto fold32 = [](float x, float y) {         // sums over the lanes 32 apart: x's in the lower half, y's in the upper
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
        return __uint_as_float(r[0]) + __uint_as_float(r[1]);
    };
    float lo = fold32(acc[0], acc[2]), hi = fold32(acc[1], acc[3]);
    const int c = 4 * c4 + 2 * (lane >> 5);
    if constexpr (LPR == 32) {
        s_acc[wave][c] = lo;
        s_acc[wave][c + 1] = hi;
    } else {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(lo), __float_as_uint(hi), false, false);
        float one = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        if (LPR == 8) one += dpp_of<0x128>(one);          // row_ror:8
        s_acc[wave][c + ((lane >> 4) & 1)] = one;
    }
    __syncthreads();
    if (tid < CH) {
        float A = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) A += s_acc[w][tid];
        const float out = W > 0.0f ? A / W : 0.0f;
        const int64_t to = b * a.o_b + (int64_t)h * a.o_h + blockIdx.z * CH + tid;
        if (a.o16) a.o16[to] = f32_to_bf16_any(out);
        else a.o[to] = out;
        if (tid == 0 && blockIdx.z == 0) a.lse[b * a.lse_b + h] = W > 0.0f ? top + __logf(W) : -INFINITY;
    }
}

int fold_states(const float* al, int64_t al_b, int64_t al_h, int64_t al_s, const StateLse& states, int slots, int sure,
                void* o, bool o_bf16, int64_t o_b, int64_t o_h, float* lse, int64_t lse_b, int B, int Hq, int D,
                void* stream) {
    if (B <= 0 || Hq <= 0 || slots < 1 || slots > 512 + kTailParts || (D != 64 && D != 128) || !al || !o || !lse || !states.p ||
        (reinterpret_cast<uintptr_t>(al) & 15) || al_b % 4 || al_h % 4 || al_s % 4 || al_s < 0 || al_s > 4096 || states.s < 0 ||
        states.s > 4096) {
        set_error("fold_states: bad shape or misaligned states");
        return -1;
    }
    const FoldArgs a{al, al_b, al_h, al_s, states.p, states.b, states.h, states.s, o_bf16 ? nullptr : static_cast<float*>(o),
                     o_bf16 ? static_cast<uint16_t*>(o) : nullptr, o_b, o_h, lse, lse_b, slots, std::min(std::max(sure, 1), slots)};
    hipStream_t st = static_cast<hipStream_t>(stream);
    // Small workgroups once there is one head per compute unit (48 requests of 32 q heads 53.5 us as one of 256 threads a head,
    // 54.7 / 57.4 as two / four, 65 with 1024 threads); below that two a head, and with many states four of 512 threads, so
    // that no thread has more than a few loads (one request of 64 K 31.7 us; 32.2 as two of 1024, 33.4 as two of 256).
    const int heads = B * Hq;
#define OMMX_FOLD(DD, Q, NT) hipLaunchKernelGGL((fold_kernel<DD, Q, NT>), dim3(B, Hq, Q), dim3(NT), 0, st, a)
    if (slots <= 96) {
        if (D == 64) OMMX_FOLD(64, 1, 256);
        else if (heads < 256) OMMX_FOLD(128, 2, 256);
        else OMMX_FOLD(128, 1, 256);
    } else {
        if (D == 64) OMMX_FOLD(64, 2, 512);
        else if (heads < 256) OMMX_FOLD(128, 4, 512);
        else OMMX_FOLD(128, 2, 512);
    }
#undef OMMX_FOLD
    if (hipGetLastError() != hipSuccess) { set_error("fold_states: launch failed"); return -2; }
    return 0;
}

template <bool HIST, bool SHARED>
static int launch_combine_rows(const CombineArgs& a, int D, hipStream_t st) {
    if (a.S > 512) return -1;
    // Pieces per head.  At batch 1 the kernel is latency bound and 2 pieces measured best (1.4 us
    // per step at 64K less than one, the same as four, 0.5 us less than eight); with many
    // (request, head) pairs the grid fills the chip by itself and one piece repeats no work.
    const bool split2 = a.B * a.Hq < 256;
    const dim3 grid(a.B, a.Hq, split2 ? 2 : 1);
    const bool small = !split2 && a.S <= 64;
    const int R = a.Hq / a.Hkv;
    // a whole kv head per workgroup once those alone are one per compute unit (32 requests of 8 kv
    // heads: 10 against 16 us; 128 requests: 25 against 47 us; with fewer, one workgroup per q head
    // spreads the work better: 16 requests 9.8 against 13 us)
    if (small && (R == 4 || R == 8) && a.Hq == R * a.Hkv && a.B * a.Hkv >= 256) {
        const dim3 g2(a.B, a.Hkv);
        const bool early = a.B * a.Hkv <= 320;       // about one workgroup per compute unit
#define OMMX_GROUPED(DD, RR)                                                                              \
        do {                                                                                              \
            if (early) hipLaunchKernelGGL((combine_grouped_kernel<DD, RR, true, HIST, SHARED>), g2, dim3(512), 0, st, a);  \
            else hipLaunchKernelGGL((combine_grouped_kernel<DD, RR, false, HIST, SHARED>), g2, dim3(512), 0, st, a);       \
        } while (0)
        if (D == 128 && R == 4) OMMX_GROUPED(128, 4);
        else if (D == 128) OMMX_GROUPED(128, 8);
        else if (D == 64 && R == 4) OMMX_GROUPED(64, 4);
        else if (D == 64) OMMX_GROUPED(64, 8);
        else return -1;
#undef OMMX_GROUPED
        return 0;
    }
    if (a.S > 256) {        // 257..512 splits: the same kernel with twice the split slots per thread
        const dim3 g1(a.B, a.Hq, split2 ? 2 : 1);
        if (D == 128 && split2) hipLaunchKernelGGL((combine_kernel<128, 2, HIST, SHARED, 1024, 512>), g1, dim3(1024), 0, st, a);
        else if (D == 128) hipLaunchKernelGGL((combine_kernel<128, 1, HIST, SHARED, 1024, 512>), g1, dim3(1024), 0, st, a);
        else if (D == 64 && split2) hipLaunchKernelGGL((combine_kernel<64, 2, HIST, SHARED, 1024, 512>), g1, dim3(1024), 0, st, a);
        else if (D == 64) hipLaunchKernelGGL((combine_kernel<64, 1, HIST, SHARED, 1024, 512>), g1, dim3(1024), 0, st, a);
        else return -1;
        return 0;
    }
    if (D == 128 && split2) hipLaunchKernelGGL((combine_kernel<128, 2, HIST, SHARED>), grid, dim3(1024), 0, st, a);
    else if (D == 128 && small) hipLaunchKernelGGL((combine_kernel<128, 1, HIST, SHARED, 512, 64>), grid, dim3(512), 0, st, a);
    else if (D == 128) hipLaunchKernelGGL((combine_kernel<128, 1, HIST, SHARED>), grid, dim3(1024), 0, st, a);
    else if (D == 64 && split2) hipLaunchKernelGGL((combine_kernel<64, 2, HIST, SHARED>), grid, dim3(1024), 0, st, a);
    else if (D == 64 && small) hipLaunchKernelGGL((combine_kernel<64, 1, HIST, SHARED, 512, 64>), grid, dim3(512), 0, st, a);
    else if (D == 64) hipLaunchKernelGGL((combine_kernel<64, 1, HIST, SHARED>), grid, dim3(1024), 0, st, a);
    else return -1;
    return 0;
}

int launch_combine(const CombineArgs& a, int D, hipStream_t st) {
    if (a.share_count)
        return a.hist_seq ? launch_combine_rows<true, true>(a, D, st) : launch_combine_rows<false, true>(a, D, st);
    return a.hist_seq ? launch_combine_rows<true, false>(a, D, st) : launch_combine_rows<false, false>(a, D, st);
}

}  // namespace ommx
