// Entry points of libommx_hip.so that only the native half of the Python launchers uses: not part of the
// C ABI.  Plain C++ (no device code), so that the host module can include it.
#pragma once
#include <stdint.h>

#define OMMX_STORE_ERR_WORDS 16

namespace ommx {

// ommx_store_pack (the C ABI documents the arguments) with one more choice: err_words, err_flag is an array of
// OMMX_STORE_ERR_WORDS host-visible ints, one per error bit.
int store_pack(const void* K, const void* V, int in_dtype, int64_t k_ts, int64_t k_hs, int64_t v_ts, int64_t v_hs,
               const int32_t* src_rows, int T, int H, int D, int page_size, int k_outliers, int index_repr,
               int select_abs, int scale_mode, int group_tokens, int group_channels, int v_bf16,
               const int32_t* dst_pages, const int32_t* dst_groups, const float* table, uint8_t* k_base,
               void* k_scale, uint16_t* k_zp, uint16_t* k_ms, uint16_t* k_mc, uint8_t* k_index, uint8_t* k_oval,
               uint8_t* v_main, void* v_scale, uint16_t* v_zp, int32_t* err_flag, bool err_words, void* stream);

// req_to_token[i] = i for i < n_pages and req_to_group[i] = i for i < n_groups, one launch.
int identity_tables(int32_t* req_to_token, int n_pages, int32_t* req_to_group, int n_groups, void* stream);

// Rows [0, n_head) and [lo, T) of a K/V block [T, H, D] (fp32 or bf16, last axis contiguous) into the history
// [hist_rows, H, D] of one request, at the ring slots of the absolute positions pos0 + row; rounds fp32 as
// torch does.  The caller has checked that every slot lies inside the history.
int rows_write(const void* K, const void* V, bool k_f32, bool v_f32, int64_t k_ts, int64_t k_hs, int64_t v_ts,
               int64_t v_hs, uint16_t* k_hist, uint16_t* v_hist, int64_t pos0, int n_head, int lo, int T, int H,
               int D, int sink, int span, void* stream);

// Up to kUploadWords 32-bit words from the host to dst inside a kernel's own argument block: no staging buffer, no
// copy engine, nothing to keep alive after the call.
constexpr int kUploadWords = 960;
int upload_words(int32_t* dst, const int32_t* host_words, int n, void* stream);

// Index tables of one store launch that packs `n` groups of a pool, from (request, group) pairs in host memory:
// src_rows[n * gt] flat history rows through the ring map, dst_pages[n * ppg], dst_groups[n].
int pack_list(const int32_t* host_pairs, int n, int32_t* src_rows, int32_t* dst_pages, int32_t* dst_groups, int gt,
              int ppg, int hist_rows, int sink, int span, int window_sink, int groups_per_seq, int pages_per_seq,
              void* stream);

// Split combine with the tail rows read in place from a bf16 row history [requests, rows, Hkv, D]: positions
// [0, min(win_sink, seq)) ++ [boundary, seq) of every request through the ring map, boundary being what
// ommx_tail_gather computes without a lag.  Saves the gather launch and the gathered copy.  o is fp32, or bf16
// rounded as torch does.
struct HistTail {
    const uint16_t *k, *v;
    int64_t stride_req;             // elements between the histories of two requests
    int rows;
    const int64_t *seq, *slots;     // device: [B] lengths, [B] history of each request (NULL: b)
    int ring_sink, ring_span, win_sink, win_recent;
};
int decode_combine_hist(const float* attn_logits, int64_t al_b, int64_t al_h, int64_t al_s, const uint16_t* q,
                        int64_t q_b, int64_t q_h, const HistTail& tail, void* o, bool o_bf16, int64_t o_b, int64_t o_h,
                        float* lse, int64_t lse_b, int B, int Hq, int Hkv, int D, int num_splits, int group_tokens,
                        float sm_scale, float logit_cap, void* stream);

// Causal attention of B requests' prompt rows over their own K/V, rows host_starts[b] .. host_starts[b + 1] of
// q [n, Hq, D], k / v [n, Hkv, D] (bf16, head_dim 64 or 128, 16-byte aligned rows, strides in elements); o fp32 or
// bf16.  Weights of fp32 precision (csrc/ommx_prefill.hip).
int prefill_attention(const uint16_t* q, int64_t q_t, int64_t q_h, const uint16_t* k, int64_t k_t, int64_t k_h,
                      const uint16_t* v, int64_t v_t, int64_t v_h, void* o, bool o_bf16, int64_t o_t, int64_t o_h,
                      const int64_t* host_starts, int B, int Hq, int Hkv, int D, float scale, void* stream);

}  // namespace ommx
