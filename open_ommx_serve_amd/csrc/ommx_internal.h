// Entry points of libommx_hip.so that only the native half of the Python launchers uses: not part of the
// C ABI.  Plain C++ (no device code), so that the host module can include it.
#pragma once
#include <stdint.h>

#define OMMX_STORE_ERR_WORDS 16

namespace ommx {

// Rows of a prompt block and their places in the history of one request (ommx_rows.h copies them).
struct BlockRows {
    const void *K, *V;
    int k_f32, v_f32, k_vec, v_vec;
    int64_t k_ts, k_hs, v_ts, v_hs;
    uint16_t *k_hist, *v_hist;
    int64_t pos0;
    int n_head, lo, H, D, sink, span;
    int rows;               // [0, n_head) and [lo, T) of the block
};

inline bool rows_aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }
inline BlockRows block_rows(const void* K, const void* V, bool k_f32, bool v_f32, int64_t k_ts, int64_t k_hs, int64_t v_ts,
                            int64_t v_hs, uint16_t* k_hist, uint16_t* v_hist, int64_t pos0, int n_head, int lo, int T,
                            int H, int D, int sink, int span) {
    const bool dst_ok = rows_aligned16(k_hist) && rows_aligned16(v_hist);
    return {K, V, k_f32, v_f32, dst_ok && rows_aligned16(K) && k_ts % 8 == 0 && k_hs % 8 == 0,
            dst_ok && rows_aligned16(V) && v_ts % 8 == 0 && v_hs % 8 == 0, k_ts, k_hs, v_ts, v_hs, k_hist, v_hist, pos0,
            n_head, lo, H, D, sink, span, n_head + (T - lo)};
}

// Groups whose rows lie in a ring history, as arguments of the store launch: the first row of each (of the flat history),
// the token at which its rows continue at the start of the ring (32 or more: none does), its destination.
struct RingGroup { int32_t row, turn, group; };
constexpr int kRingGroups = 96;
struct RingGroups { RingGroup of[kRingGroups]; };

// The new rows of a decode step (ring_step below): pool slots, positions and packed lengths of its requests.
constexpr int kStepRows = 64;
struct StepRows { int32_t slot[kStepRows], pos[kStepRows], packed[kStepRows]; };
// The same rows written by the store launch that packs the groups complete with them: rows of K and V, histories [slots, rows, H, D],
// all 16 bytes at a time.  None of the groups reads a row that the step writes.
struct StepWrite {
    const uint16_t *k, *v;
    int64_t k_bs, k_hs, v_bs, v_hs;
    uint16_t *k_hist, *v_hist;
    int64_t stride_req;
    int32_t *block, *err;
    int B, H, rows, sink, span;
    StepRows at;
};

// What a store launch of the native launchers does besides packing.
struct StoreExtras {
    bool err_words = false;               // err_flag is an array of OMMX_STORE_ERR_WORDS host-visible ints, one per error bit
    int32_t *own_pages = nullptr, *own_groups = nullptr;      // identity tables [T / page_size], [T / group_tokens] to
                                                              // fill (both or neither)
    const StepWrite* step = nullptr;      // with `ring`: rows to write beside them
    const RingGroups* ring = nullptr;     // where the groups lie; T / 32 of them, span rows in the ring.  store_pack returns 1,
    int ring_span = 0;                    // with nothing launched, for a recipe or a number of groups that needs the tables
    const BlockRows* rows = nullptr;      // bf16 rows to copy into the history (head_dim a multiple of 8, every slot inside it),
                                          // at most kRowSlices for a group
};
// The rows of StoreExtras are slices of the grid's y or z behind those of the groups, a row for every group in a slice: few
// groups under a long recent window would need more slices than a grid has (65 536).
constexpr int64_t kRowSlices = 32768;

// ommx_store_pack (the C ABI documents the arguments) with extras.
int store_pack(const void* K, const void* V, int in_dtype, int64_t k_ts, int64_t k_hs, int64_t v_ts, int64_t v_hs,
               const int32_t* src_rows, int T, int H, int D, int page_size, int k_outliers, int index_repr,
               int select_abs, int scale_mode, int group_tokens, int group_channels, int v_bf16,
               const int32_t* dst_pages, const int32_t* dst_groups, const float* table, uint8_t* k_base,
               void* k_scale, uint16_t* k_zp, uint16_t* k_ms, uint16_t* k_mc, uint8_t* k_index, uint8_t* k_oval,
               uint8_t* v_main, void* v_scale, uint16_t* v_zp, int32_t* err_flag, const StoreExtras& extras,
               void* stream);

// The rows in one launch; fp32 is rounded as torch does.  The caller has checked that every slot lies inside the history.
int rows_write(const BlockRows& rows, void* stream);

// Prompts of several fresh requests that lie behind one another in K / V [rows, H, D] (bf16): every row into its request's
// whole history (no ring), and the index tables of the one store launch that packs all their groups.
struct PromptBlocks {
    const uint16_t *K, *V;
    int64_t k_ts, k_hs, v_ts, v_hs;
    uint16_t *k_hist, *v_hist;
    int64_t stride_req;             // elements between the histories of two requests
    int H, D, window_sink, gt, ps, groups_per_seq;
};
constexpr int kPromptsPerLaunch = 240;
// {first row in K, row behind the last, slot, groups before this request's} of each request
struct PromptRow { int32_t first, end, slot, group0; };
// prompts[n], in the order of their rows; groups[n] groups of each; src_rows / dst_pages / dst_groups as ommx_store_pack
// takes them, all groups together.
int prompt_blocks(const PromptBlocks& blocks, const PromptRow* prompts, int n, int32_t total_groups, int32_t* src_rows,
                  int32_t* dst_pages, int32_t* dst_groups, void* stream);

// Up to kUploadWords 32-bit words from the host to dst inside a kernel's own argument block: no staging buffer, no
// copy engine, nothing to keep alive after the call.
constexpr int kUploadWords = 960;
int upload_words(int32_t* dst, const int32_t* host_words, int n, void* stream);
// int64 [write position | length | tail positions], n64 of them, then int32 [packed length | tail rows]
int step_block(int32_t* block, int n64, int64_t seq, int64_t boundary, int sink, int tail, int packed, void* stream);

// One new row of every request of a step into its ring history, slots and positions as arguments of the launch; `block`
// (may be NULL) receives what later launches of the step read on the device: int64 slots[B], positions[B], lengths after
// the step[B], then int32 packed lengths[B].
int ring_step(const uint16_t* k, const uint16_t* v, int64_t k_bs, int64_t k_hs, int64_t v_bs, int64_t v_hs, uint16_t* k_hist,
              uint16_t* v_hist, int64_t stride_req, int rows, int B, int H, int D, int sink, int span, const StepRows& step,
              int32_t* block, int32_t* err, void* stream);

// Index tables of one store launch that packs `n` groups of a pool, from (request, group) pairs in host memory:
// src_rows[n * gt] flat history rows through the ring map, dst_pages[n * ppg], dst_groups[n].
int pack_list(const int32_t* host_pairs, int n, int32_t* src_rows, int32_t* dst_pages, int32_t* dst_groups, int gt,
              int ppg, int hist_rows, int sink, int span, int window_sink, int groups_per_seq, int pages_per_seq,
              void* stream);

// Where the log-sum-exp of the split states lies when it is not column D of the states.
struct StateLse { float* p; int64_t b, h, s; };

// The packed groups of the whole batch dealt out in equal pieces (csrc/ommx_decode_shares.h) instead of num_splits per
// request: at most `all` of them (`few`, if a third resident workgroup per compute unit does not pay), at most
// num_splits for one request, single groups while the batch has no more than `singles`.  `each` is about what one of B requests of the same length gets;
// count int32[B] receives
// the number of pieces of every request, which the combine entries take.
struct Shares { int all, few, singles, each; int32_t* count; };

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
                        float sm_scale, float logit_cap, const StateLse& states, const Shares* shares, void* stream);

// The bf16 tail rows as kTailParts more states of every (request, q head), attended by the split-KV launch itself: slots
// 0 .. kTailParts - 1 of the state rows, in front of the splits' own (attn_logits and the lse plane point behind them).
// Gathered rows (tail lengths) or rows of a history (seq), as above.  K and V rows 16-byte aligned.
constexpr int kTailParts = 4;
struct DecodeTail {
    const uint16_t *kt, *vt;
    int64_t kt_b, kt_t, kt_h, vt_b, vt_t, vt_h;
    const int32_t* tail;            // gathered: rows of every request, at most T (0: not told)
    int T;
    const int64_t *hist_seq, *hist_slots;
    int hist_rows, ring_sink, ring_span, win_sink, win_recent, gt;
};

// o and lse of every (request, q head) from its `slots` states (rows of D floats, lse plane beside them): the merge when
// the tail rows are among the states.  `sure`: how many slots are read before their lse is known.
int fold_states(const float* al, int64_t al_b, int64_t al_h, int64_t al_s, const StateLse& states, int slots, int sure,
                void* o, bool o_bf16, int64_t o_b, int64_t o_h, float* lse, int64_t lse_b, int B, int Hq, int D,
                void* stream);

// What the kernel for short calls (csrc/ommx_decode_team.hip) is told beyond the common arguments: entries of a row of either table,
// 32-token groups of a split (fixed splits), and the merge, when the launch does it itself (up to kTeamMerged splits or shares of a
// request): `arrivals`, a word every 64 bytes for each (request, kv head or pair of 64-channel ones), memory that only this call uses,
// whatever it holds; `number` of this call, from kFirstCall on and below 2^56, no two the same (so not in a launch that is replayed).
constexpr uint64_t kFirstCall = 0xFF000000000000ull;
constexpr int kTeamMerged = 32;
struct TeamMerge {
    int rt_n, rg_n, per_split;
    float* o; uint16_t* o16;        // one of them
    int64_t o_b, o_h;
    float* lse; int64_t lse_b;
    unsigned long long* arrivals;   // NULL: states only
    uint64_t number;
};

// ommx_decode_splitkv / _ref (plain) with these choices (each may be NULL).  Returns 1, with nothing done, when shares
// are asked for and no kernel with shares serves the call.  *tail_done tells whether the launch attends the tail.  team: by the
// kernel for short calls (csrc/ommx_decode_team.hip); returns 1, with nothing done, for what it does not serve.
#define OMMX_DECODE_DECL                                                                            \
    const uint16_t* q, int64_t q_stride_b, int64_t q_stride_h, const uint8_t* k_base,               \
    const void* k_scale, const uint16_t* k_zp, const uint16_t* k_ms, const uint16_t* k_mc,          \
    const uint8_t* k_index, const uint8_t* k_oval, const uint8_t* v_main, const void* v_scale,      \
    const uint16_t* v_zp, const void* req_to_token, int64_t rt_stride, const void* req_to_group,    \
    int64_t rg_stride, int table_i64, const int32_t* b_seq_len, float* attn_logits,                 \
    int64_t al_stride_b, int64_t al_stride_h, int64_t al_stride_s, int B, int Hq, int Hkv, int D,   \
    int page_size, int k_outliers, int index_repr, int scale_bf16, int group_tokens,                \
    int group_channels, int v_bf16, int num_splits, float sm_scale, float logit_cap,                \
    int packed_start_offset, int seg_group_base, int num_pages, int num_group_slots,                \
    int32_t* err_flag, void* stream
int decode_splitkv(OMMX_DECODE_DECL, bool plain, const StateLse* lse, const Shares* shares, const DecodeTail* tail,
                   bool* tail_done, const TeamMerge* team = nullptr);
#undef OMMX_DECODE_DECL

// ommx_decode_combine with the lse of the states elsewhere (NULL: column D) and the shares they come from (NULL:
// num_splits states per request; else at most that many).
int decode_combine(const float* attn_logits, int64_t al_b, int64_t al_h, int64_t al_s, const uint16_t* q, int64_t q_b,
                   int64_t q_h, const uint16_t* k_tail, const uint16_t* v_tail, int64_t kt_b, int64_t kt_t, int64_t kt_h,
                   int64_t vt_b, int64_t vt_t, int64_t vt_h, const int32_t* b_tail_len, const int32_t* b_seq_len,
                   float* o, int64_t o_b, int64_t o_h, float* lse, int64_t lse_b, int B, int Hq, int Hkv, int D,
                   int num_splits, int group_tokens, int tail_rows, float sm_scale, float logit_cap,
                   const StateLse* states, const Shares* shares, void* stream);

// Causal attention of B requests' prompt rows over their own K/V, rows host_starts[b] .. host_starts[b + 1] of
// q [n, Hq, D], k / v [n, Hkv, D] (bf16, head_dim 64 or 128, 16-byte aligned rows, strides in elements); o fp32 or
// bf16.  Weights of fp32 precision (csrc/ommx_prefill.hip).  A 64-key tile of K and of V is addressed by 32-bit byte
// offsets, which bounds their row strides; a bit per tile of the longest request fits the kernel's LDS.
constexpr int64_t kPrefillMaxStride = 1 << 24;
constexpr int kPrefillMaxRows = 1 << 18;
// The form of the kernel that a batch takes: a group of waves a workgroup, two that share the keys of its rows, two with rows each.
enum class PrefillForm { one_group, split_keys, two_groups };
PrefillForm prefill_form(const int64_t* host_starts, int B, int Hq, int D);
int prefill_attention(const uint16_t* q, int64_t q_t, int64_t q_h, const uint16_t* k, int64_t k_t, int64_t k_h,
                      const uint16_t* v, int64_t v_t, int64_t v_h, void* o, bool o_bf16, int64_t o_t, int64_t o_h,
                      const int64_t* host_starts, int B, int Hq, int Hkv, int D, float scale, void* stream);

}  // namespace ommx
