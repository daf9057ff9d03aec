// Argument block and small helpers shared by the decode kernels.
#pragma once
#include "ommx_common.h"
#include "ommx_internal.h"

namespace ommx {

struct DecodeArgs {
    const uint16_t* q; int64_t q_sb, q_sh;
    const uint8_t* k_base; const int8_t* k_scale; const uint16_t* k_zp;
    const uint16_t* k_ms; const uint16_t* k_mc;
    const uint8_t* k_obmp;           // index plane: 4-byte bitmaps, or 7-bit position streams (idx_repr 1)
    const uint8_t* k_oval;
    const uint8_t* v_main; const int8_t* v_scale; const uint16_t* v_zp;
    const void* rt; int64_t rt_s; const void* rg; int64_t rg_s; int i64;
    const int32_t* seq;
    float* al; int64_t al_b, al_h, al_s;
    int B, Hq, Hkv, ps, kout, S;
    float sm_scale, cap;
    int off, gbase;
    int idx_repr;                    // 0 flat bitmap, 1 relidx7
    int scale_bf16;                  // k_scale / v_scale hold bf16 steps instead of int8 exponents
    int gt, gc;                      // tokens per K group, channels per V vector (16, 32, 64 or 128)
    int v_bf16;                      // v_main holds bf16 rows [P,ps,H,D] instead of INT2 codes
    // Extents of the planes the tables index: a page id outside [0, n_pages) or a group slot outside
    // [0, n_gslots) is clamped into range (no access leaves the planes) and OMMX_ERR_TABLE_RANGE is
    // OR-ed into *err (may be NULL).  0 = extent not given: ids are used as they are.
    int n_pages, n_gslots;
    int32_t* err;
    // Where the lse of a state goes: attn_logits' column D of the C ABI, or a plane of its own (the caller's workspace
    // has rows of D + 1; in a workspace of our own the rows are D floats, aligned, and the merge reads the lse of all
    // states of a head from a few cache lines).
    float* sl; int64_t sl_b, sl_h, sl_s;
    // Work dealt out in shares instead of a fixed number of splits per request (ommx_decode_shares.h): workgroups along
    // x with a third resident workgroup per compute unit and without, the most groups of a batch that get a share
    // each, and where the kernel leaves the number of shares of every request (at most S) for the combine.
    // shares 0: fixed splits.
    int shares, shares_few, singles;
    int32_t* share_count;
    // set by the launcher of the serving-recipe kernel only: head_dim is 64 and Hkv counts PAIRS of kv
    // heads (the planes of two neighbouring 64-channel heads read like one 128-channel head)
    int half;
    // The tail rows attended by this launch (ommx_decode_tail.h): that many workgroups more per head group, 0 none, at the
    // end of the grid: slices of z behind the requests, or of y behind the shares.
    int t_slices;
    DecodeTail t;
};

// 7-bit position streams (pack.py:128-164): position s of a frame at bits [7s, 7s+7)
__host__ __device__ constexpr int relidx7_bytes(int k) { return (7 * k + 7) / 8; }

__device__ __forceinline__ int64_t table_at(const void* t, int64_t i, int i64) {
    return i64 ? static_cast<const int64_t*>(t)[i] : static_cast<const int32_t*>(t)[i];
}

// Page id / group slot as read from a table, held inside the plane; `bad` collects whether any was not.
__host__ __device__ __forceinline__ int clamp_id(int id, int n, bool& bad) {
    if (n > 0) {
        const uint32_t u = static_cast<uint32_t>(id), top = static_cast<uint32_t>(n - 1);
        bad |= u > top;                       // negative ids are huge as unsigned: one comparison
        id = static_cast<int>(u < top ? u : top);
    }
    return id;
}
__device__ __forceinline__ void report_table_range(int32_t* err, bool bad) {
    if (__any(bad) && err && (threadIdx.x & 63) == 0) atomicOr(err, OMMX_ERR_TABLE_RANGE);
}

__device__ __forceinline__ float apply_cap(float x, float cap) {
    // cap * tanh(x / cap) written as the reference does: cap * (2*sigmoid(2x/cap) - 1)
    if (cap > 0.0f) x = cap * (2.0f / (1.0f + __expf(-2.0f * x / cap)) - 1.0f);
    return x;
}


struct CombineArgs {
    const float* al; int64_t al_b, al_h, al_s;
    const uint16_t* q; int64_t q_sb, q_sh;
    const uint16_t* kt; const uint16_t* vt;
    int64_t kt_b, kt_t, kt_h, vt_b, vt_t, vt_h;
    const int32_t* tail; const int32_t* seq;
    float* o; int64_t o_b, o_h;
    float* lse; int64_t lse_b;
    int B, Hq, Hkv, S;
    float sm_scale, cap;
    int gt;                          // tokens per K group: the splits are rounded to it
    int T;                           // rows every request's tail buffer holds (0: not told): rows below it
                                     // may be read before b_tail_len has arrived
    const float* sl; int64_t sl_b, sl_h, sl_s;      // lse of the states, as in DecodeArgs
    uint16_t* o16;                   // bf16 output in place of o (same strides); NULL: fp32 into o
    // Tail rows read in place from the row history instead of a gathered buffer: kt / vt are the histories, kt_b
    // the elements between two requests' histories, and the rows follow from the sequence length (TailRows below).
    const int64_t* hist_seq;         // NULL: gathered buffer
    const int64_t* hist_slots;       // NULL: request b uses history b
    int hist_rows, ring_sink, ring_span, win_sink, win_recent;
    const int32_t* share_count;      // states of every request (at most S); NULL: S each
    int sure;                        // state slots to read before share_count is here (S without it)
};

// The bf16 rows of one request: how many, and where row t of them lies (elements from the K / V base pointers).
// Gathered buffer: rows 0, 1, ... of the request.  History: positions [0, min(sink, seq)) ++ [boundary, seq)
// (kv_pool.py:1080-1097) through the ring map of kv_store.py:301-327; the sliding part starts at ring offset
// `turn`, so a row costs one conditional subtraction instead of a remainder.
template <bool HIST>
struct TailRows {
    int n, n_sink, turn, span, sink, cap;
    int64_t k_base, v_base;

    // A: CombineArgs or DecodeTail
    template <class A>
    __device__ __forceinline__ void init(const A& a, int b) {
        if constexpr (!HIST) {
            // a length outside the tail buffer (when the caller has said how many rows it holds) is held
            // inside it, so that no row address leaves the buffer whatever b_tail_len contains
            n = a.tail ? a.tail[b] : 0;
            n = max(n, 0);
            if (a.T > 0) n = min(n, a.T);
            k_base = b * a.kt_b;
            v_base = b * a.vt_b;
            return;
        }
        const int seq = static_cast<int>(a.hist_seq[b]), slot = a.hist_slots ? static_cast<int>(a.hist_slots[b]) : b;
        k_base = slot * a.kt_b;
        v_base = slot * a.vt_b;
        const int extra = seq - a.win_sink - a.win_recent;
        n_sink = min(seq, a.win_sink);
        const int boundary = extra <= 0 ? n_sink : a.win_sink + extra / a.gt * a.gt;
        n = min(max(0, n_sink + max(seq - boundary, 0)), a.T);
        sink = a.ring_sink;
        span = a.ring_span;
        cap = a.hist_rows;
        turn = span > 0 && boundary >= sink ? (boundary - sink) % span : boundary - sink;
    }
    __device__ __forceinline__ int row(int t) const {
        if constexpr (!HIST) return t;
        if (t < n_sink) return t;              // (the ring pins the window's sink rows: ring_sink == win_sink, or no ring)
        int r = turn + (t - n_sink);
        if (span > 0 && r >= span) r -= span;
        r += sink;
        return min(max(r, 0), cap - 1);
    }
};

int launch_decode_ref(const DecodeArgs& a, int D, int R, hipStream_t st);
int launch_combine(const CombineArgs& a, int D, hipStream_t st);

}  // namespace ommx
