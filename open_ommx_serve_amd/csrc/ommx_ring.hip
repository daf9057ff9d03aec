// bf16 residual ring of the KV store: the rows that are not (yet) packed.
//
//   ring_write_kernel   one new K/V row per request into its ring slot (ring_step_kernel: places as arguments); follows
//                       ommx_gpu_serve/attention/kv_store_ops.py:22-40 (_kv_write_token) and
//                       the batched scatter of attention/kv_pool.py:407-419.
//   tail_gather_kernel  sink + recent rows of every request into the fixed tail buffers,
//                       with the window arithmetic of attention/kv_pool.py:1048-1105
//                       (decode_inputs_device) done in the kernel from the device sequence
//                       lengths; or, given explicit positions, the plain gather of
//                       kv_store_ops.py:42-61 (_kv_gather_tail).
//
// Ring slot of absolute position p (kv_store.py:301-327): p below the sink count stays,
// everything else slides modulo the ring span: sink + (p - sink) % span.  span == 0 means
// the history is kept whole and the slot is the position.
//
// Both kernels are pure row copies (H*D bf16 per row), 16 bytes per thread when rows are
// 16-byte aligned, one workgroup per row.  A step's write is a few rows: its time is a launch and a chain of memory
// latencies, so the new row is asked for beside its position (8 heads of 128: one piece of K or V a thread), and a thread's
// piece and head are its numbers: found by a division of one number, one request 1.58 us instead of 1.44, 8 requests 2.54
// instead of 2.44.
#include <algorithm>

#include "ommx_ring_args.h"
#include "ommx_rows.h"

namespace ommx {

// Copies n_elem bf16 from src (rows of D contiguous elements, head stride hs) to a dense row.
__device__ __forceinline__ void copy_row_in(uint16_t* dst, const uint16_t* src, int64_t hs,
                                            int H, int D, bool vec) {
    if (vec) {
        const int per_head = D / 8;
        for (int i = threadIdx.x; i < H * per_head; i += blockDim.x) {
            const int h = i / per_head, c = (i % per_head) * 8;
            *reinterpret_cast<uint4*>(dst + h * D + c) =
                *reinterpret_cast<const uint4*>(src + h * hs + c);
        }
    } else {
        for (int i = threadIdx.x; i < H * D; i += blockDim.x) dst[i] = src[(i / D) * hs + i % D];
    }
}

// Thread (x, y) of a workgroup copies the piece of eight x of head y of a new row of K, of head y - H of V, and of every
// blockDim.y-th head after that.
__device__ __forceinline__ uint4 new_row_piece(const RingArgs& a, const uint16_t* k, const uint16_t* v, int64_t k_bs,
                                               int64_t k_hs, int64_t v_bs, int64_t v_hs, int b, int y) {
    const bool is_v = y >= a.H;
    return *reinterpret_cast<const uint4*>((is_v ? v + b * v_bs + (y - a.H) * v_hs : k + b * k_bs + y * k_hs) + 8 * threadIdx.x);
}
// Row b of K and V to position p of history `slot`; `first` is the thread's first piece.
__device__ __forceinline__ void put_new_row(const RingArgs& a, const uint16_t* k, const uint16_t* v, int64_t k_bs, int64_t k_hs,
                                            int64_t v_bs, int64_t v_hs, int b, int64_t p, int64_t slot, bool vec, uint4 first) {
    const int64_t row = ring_slot(p, a.sink, a.span);
    if (row < 0 || row >= a.cap) {         // kv_store_ops.py:33-34 asserts here
        if (a.err && (threadIdx.x | threadIdx.y) == 0) atomicOr(a.err, OMMX_ERR_RING_RANGE);
        return;
    }
    const int64_t off = slot * a.req_stride + row * (int64_t)(a.H * a.D);
    if (vec) {
        auto put = [&](int y, uint4 x) {
            const bool is_v = y >= a.H;
            *reinterpret_cast<uint4*>((is_v ? a.v_hist : a.k_hist) + off + ((is_v ? y - a.H : y) * a.D + 8 * static_cast<int>(threadIdx.x))) = x;
        };
        put(threadIdx.y, first);
        for (int y = threadIdx.y + blockDim.y; y < 2 * a.H; y += blockDim.y)
            put(y, new_row_piece(a, k, v, k_bs, k_hs, v_bs, v_hs, b, y));
        return;
    }
    copy_row_in(a.k_hist + off, k + b * k_bs, k_hs, a.H, a.D, false);
    copy_row_in(a.v_hist + off, v + b * v_bs, v_hs, a.H, a.D, false);
}

__global__ void __launch_bounds__(1024) ring_write_kernel(
    RingArgs a, const uint16_t* k, const uint16_t* v, int64_t k_bs, int64_t k_hs, int64_t v_bs,
    int64_t v_hs, const int64_t* pos, int64_t* pos_next, int vec) {
    const int b = blockIdx.x;
    uint4 first = {};
    if (vec) first = new_row_piece(a, k, v, k_bs, k_hs, v_bs, v_hs, b, threadIdx.y);
    const int64_t p = pos[b];
    const int64_t slot = a.slots ? a.slots[b] : b;
    __syncthreads();                       // every thread has read pos[b] before it moves
    if (pos_next && (threadIdx.x | threadIdx.y) == 0) pos_next[b] = p + 1;
    put_new_row(a, k, v, k_bs, k_hs, v_bs, v_hs, b, p, slot, vec, first);
}

// The same with the places as arguments: no launch before this one has to bring them to the device; the step's other launches
// read them from `block`, which the first layer's launch fills.  8 requests of 8 heads, kernel alone 2.4 us as the other, and the
// upload's 1.4 are gone; the host's part of a step of two layers without its decodes 29 -> 20 us.
__global__ void __launch_bounds__(1024) ring_step_kernel(RingArgs a, const uint16_t* k, const uint16_t* v, int64_t k_bs,
                                                         int64_t k_hs, int64_t v_bs, int64_t v_hs, int32_t* block, int vec,
                                                         StepRows step) {
    const int b = blockIdx.x, B = gridDim.x, p = step.pos[b], slot = step.slot[b];
    uint4 first = {};
    if (vec) first = new_row_piece(a, k, v, k_bs, k_hs, v_bs, v_hs, b, threadIdx.y);
    if (block && (threadIdx.x | threadIdx.y) == 0) {
        int64_t* const wide = reinterpret_cast<int64_t*>(block);
        wide[b] = slot;
        wide[B + b] = p;
        wide[2 * B + b] = p + 1LL;
        block[6 * B + b] = step.packed[b];
    }
    put_new_row(a, k, v, k_bs, k_hs, v_bs, v_hs, b, p, slot, vec, first);
}

__global__ void __launch_bounds__(256) tail_gather_kernel(
    RingArgs a, const int64_t* seq, const int64_t* tail_idx, uint16_t* k_tail, uint16_t* v_tail,
    int T, int recent, int gt, int lag, int32_t* b_tail_len, int32_t* b_seq_len, int vec) {
    const int t = blockIdx.x, b = blockIdx.y;
    int64_t abs_pos;
    if (tail_idx) {
        abs_pos = tail_idx[(int64_t)b * T + t];
    } else {
        // kv_pool.py:1080-1097: boundary, counts and the sink ++ recent position ramp.  The
        // packed boundary is the one of the length the planes were last packed for, `lag`
        // tokens ago: rows appended since then are read from the ring, the group they may
        // have completed included.
        const int64_t s = seq[b];
        const int64_t s_packed = s > lag ? s - lag : 0;
        const int64_t extra = s_packed - a.sink - recent;
        const int64_t n_sink = s < a.sink ? s : a.sink;
        const int64_t boundary = extra <= 0 ? n_sink : a.sink + (extra / gt) * gt;
        const int64_t n_rec = s > boundary ? s - boundary : 0;
        const int64_t n_total = n_sink + n_rec;
        abs_pos = t < n_sink ? t : boundary + (t - n_sink);
        if (t >= n_total) abs_pos = 0;     // padding rows repeat position 0; readers mask them
        if (t == 0 && threadIdx.x == 0) {
            if (b_tail_len) b_tail_len[b] = (int32_t)(n_total < T ? n_total : T);
            if (b_seq_len) b_seq_len[b] = (int32_t)(boundary > a.sink ? boundary - a.sink : 0);
        }
    }
    const int64_t slot = a.slots ? a.slots[b] : b;
    const int64_t row = ring_slot(abs_pos, a.sink, a.span);
    const int HD = a.H * a.D;
    uint16_t* kd = k_tail + ((int64_t)b * T + t) * HD;
    uint16_t* vd = v_tail + ((int64_t)b * T + t) * HD;
    if (row < 0 || row >= a.cap) {         // kv_store_ops.py:52-53 asserts here
        if (a.err && threadIdx.x == 0) atomicOr(a.err, OMMX_ERR_RING_RANGE);
        for (int i = threadIdx.x; i < HD; i += blockDim.x) { kd[i] = 0; vd[i] = 0; }
        return;
    }
    const uint16_t* ks = a.k_hist + slot * a.req_stride + row * (int64_t)HD;
    const uint16_t* vs = a.v_hist + slot * a.req_stride + row * (int64_t)HD;
    if (vec) {
        for (int i = threadIdx.x; i < HD / 8; i += blockDim.x) {
            reinterpret_cast<uint4*>(kd)[i] = reinterpret_cast<const uint4*>(ks)[i];
            reinterpret_cast<uint4*>(vd)[i] = reinterpret_cast<const uint4*>(vs)[i];
        }
    } else {
        for (int i = threadIdx.x; i < HD; i += blockDim.x) { kd[i] = ks[i]; vd[i] = vs[i]; }
    }
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

static bool ring_rows_vec(const RingArgs& a, const uint16_t* k, const uint16_t* v, int64_t k_bs, int64_t k_hs, int64_t v_bs,
                          int64_t v_hs) {
    return a.D % 8 == 0 && a.D <= 8192 && aligned16(a.k_hist) && aligned16(a.v_hist) && aligned16(k) && aligned16(v) &&
           a.req_stride % 8 == 0 && k_bs % 8 == 0 && k_hs % 8 == 0 && v_bs % 8 == 0 && v_hs % 8 == 0;
}
static dim3 ring_row_threads(const RingArgs& a, bool vec) {
    if (!vec) return dim3(a.H * a.D >= 256 ? 256 : 128);
    return dim3(a.D / 8, std::min(2 * a.H, 1024 / (a.D / 8)));
}

int launch_ring_write(const RingArgs& a, const uint16_t* k, const uint16_t* v, int64_t k_bs,
                      int64_t k_hs, int64_t v_bs, int64_t v_hs, const int64_t* pos,
                      int64_t* pos_next, int B, hipStream_t st) {
    const bool vec = ring_rows_vec(a, k, v, k_bs, k_hs, v_bs, v_hs);
    hipLaunchKernelGGL(ring_write_kernel, dim3(B), ring_row_threads(a, vec), 0, st, a, k, v, k_bs, k_hs, v_bs,
                       v_hs, pos, pos_next, vec);
    return 0;
}

int ring_step(const uint16_t* k, const uint16_t* v, int64_t k_bs, int64_t k_hs, int64_t v_bs, int64_t v_hs, uint16_t* k_hist,
              uint16_t* v_hist, int64_t stride_req, int rows, int B, int H, int D, int sink, int span, const StepRows& step,
              int32_t* block, int32_t* err, void* stream) {
    if (B < 1 || B > kStepRows || H < 1 || D < 1 || rows < 1) { set_error("ring_step: bad shape"); return -1; }
    const RingArgs a{k_hist, v_hist, stride_req, rows, sink, span, H, D, nullptr, err};
    const bool vec = ring_rows_vec(a, k, v, k_bs, k_hs, v_bs, v_hs);
    hipLaunchKernelGGL(ring_step_kernel, dim3(B), ring_row_threads(a, vec), 0, static_cast<hipStream_t>(stream), a, k, v,
                       k_bs, k_hs, v_bs, v_hs, block, vec, step);
    if (hipGetLastError() != hipSuccess) { set_error("ring_step: launch failed"); return -2; }
    return 0;
}

int launch_tail_gather(const RingArgs& a, const int64_t* seq, const int64_t* tail_idx,
                       uint16_t* k_tail, uint16_t* v_tail, int B, int T, int recent, int gt,
                       int lag, int32_t* b_tail_len, int32_t* b_seq_len, hipStream_t st) {
    const int vec = (a.H * a.D) % 8 == 0 && aligned16(a.k_hist) && aligned16(a.v_hist) &&
                    aligned16(k_tail) && aligned16(v_tail) && a.req_stride % 8 == 0;
    const int threads = (a.H * a.D / (vec ? 8 : 1)) >= 256 ? 256 : 128;
    hipLaunchKernelGGL(tail_gather_kernel, dim3(T, B), dim3(threads), 0, st, a, seq, tail_idx,
                       k_tail, v_tail, T, recent, gt, lag, b_tail_len, b_seq_len, vec);
    return 0;
}

// ---- prompt blocks ---------------------------------------------------------------------------
// One workgroup per row (ommx_rows.h).  Bound by HBM for long blocks, by the launch for a few rows; replaces one torch copy
// per tensor (whole history) or nine small index launches (ring).  A prompt that completes groups carries its live rows
// in the store launch instead.
__global__ void __launch_bounds__(256) rows_write_kernel(BlockRows a) { copy_block_row<true>(a, blockIdx.x); }

int rows_write(const BlockRows& a, void* stream) {
    if (a.D % 8 || a.n_head < 0 || a.lo < a.n_head || a.rows < a.n_head) { set_error("rows_write: bad shape"); return -1; }
    if (a.rows == 0) return 0;
    hipLaunchKernelGGL(rows_write_kernel, dim3(a.rows), dim3(a.H * a.D / 8 > 64 ? 128 : 64), 0,
                       static_cast<hipStream_t>(stream), a);
    if (hipGetLastError() != hipSuccess) { set_error("rows_write: launch failed"); return -2; }
    return 0;
}

// ---- prompts of several requests -------------------------------------------------------------
// One workgroup per row: it finds its request in the table that came with the launch (a scalar search over the first
// rows), copies the row, and its first thread notes where the row's token is packed from and to.  One launch for rows and
// lists and one store launch of all groups, instead of a row copy and a store launch per request: these grids fill the chip
// where eight prompts of 100 to 700 rows used to take 16 launches of 3.4 to 4.7 and 6.4 to 7.0 us one after another.
struct PromptTable { PromptRow row[kPromptsPerLaunch]; };
static_assert(sizeof(PromptTable) <= kUploadWords * sizeof(int32_t), "the argument block");

__global__ void __launch_bounds__(128) prompt_rows_kernel(PromptBlocks a, int n, int32_t total_groups, int32_t* src_rows,
                                                          int32_t* dst_pages, int32_t* dst_groups, int vec, PromptTable t) {
    const int row = t.row[0].first + blockIdx.x;
    int lo = 0, hi = n - 1;                        // the last request whose first row is not behind this one
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (t.row[mid].first <= row) lo = mid;
        else hi = mid - 1;
    }
    const PromptRow r = t.row[lo];
    const int pos = row - r.first;
    const int64_t to = r.slot * a.stride_req + pos * static_cast<int64_t>(a.H * a.D);
    copy_row_in(a.k_hist + to, a.K + row * a.k_ts, a.k_hs, a.H, a.D, vec);
    copy_row_in(a.v_hist + to, a.V + row * a.v_ts, a.v_hs, a.H, a.D, vec);
    const int p = pos - a.window_sink, groups = (lo + 1 < n ? t.row[lo + 1].group0 : total_groups) - r.group0;
    if (threadIdx.x == 0 && p >= 0 && p < groups * a.gt) {
        const int at = r.group0 * a.gt + p;
        src_rows[at] = row;
        if (p % a.ps == 0) dst_pages[at / a.ps] = r.slot * (a.groups_per_seq * (a.gt / a.ps)) + p / a.ps;
        if (p % a.gt == 0) dst_groups[at / a.gt] = r.slot * a.groups_per_seq + p / a.gt;
    }
}

int prompt_blocks(const PromptBlocks& a, const PromptRow* prompts, int n, int32_t total_groups, int32_t* src_rows,
                  int32_t* dst_pages, int32_t* dst_groups, void* stream) {
    if (n < 1 || n > kPromptsPerLaunch || a.gt < 1 || a.ps < 1 || a.gt % a.ps) { set_error("prompt_blocks: bad shape"); return -1; }
    PromptTable t;
    for (int i = 0; i < n; ++i) t.row[i] = prompts[i];
    const int vec = a.D % 8 == 0 && aligned16(a.k_hist) && aligned16(a.v_hist) && aligned16(a.K) && aligned16(a.V) &&
                    a.stride_req % 8 == 0 && (a.k_ts | a.k_hs | a.v_ts | a.v_hs) % 8 == 0;
    hipLaunchKernelGGL(prompt_rows_kernel, dim3(prompts[n - 1].end - prompts[0].first), dim3(128), 0,
                       static_cast<hipStream_t>(stream), a, n, total_groups, src_rows, dst_pages, dst_groups, vec, t);
    if (hipGetLastError() != hipSuccess) { set_error("prompt_blocks: launch failed"); return -2; }
    return 0;
}

// ---- small host-to-device blocks through the kernel argument buffer ----------------------------
// A host-to-device copy of a few hundred bytes of pageable memory costs 10-15 us of host time and waits for its
// staging; a launch that carries the words as its arguments costs 2 us and leaves nothing behind.
struct Words { int32_t w[kUploadWords]; };

__global__ void __launch_bounds__(256) upload_words_kernel(int32_t* dst, int n, Words words) {
    for (int i = threadIdx.x; i < n; i += 256) dst[i] = words.w[i];
}

int upload_words(int32_t* dst, const int32_t* host_words, int n, void* stream) {
    Words w;
    for (int done = 0; done < n; done += kUploadWords) {
        const int m = n - done < kUploadWords ? n - done : kUploadWords;
        for (int i = 0; i < m; ++i) w.w[i] = host_words[done + i];
        hipLaunchKernelGGL(upload_words_kernel, dim3(1), dim3(256), 0, static_cast<hipStream_t>(stream),
                           dst + done, m, w);
    }
    if (hipGetLastError() != hipSuccess) { set_error("upload_words: launch failed"); return -2; }
    return 0;
}

// The block of a one-request step: int64 write position, length and positions of the tail rows (the first `sink`, then those from
// `boundary` on, `tail` in all, zeros behind them), int32 packed length and tail count.  The positions follow from four numbers: as a list
// made on the host and sent as words they were 5 us of a step's 11 there (3.2 of them the launch, which takes as long on the GPU).
__global__ void __launch_bounds__(256) step_block_kernel(int64_t* wide, int n64, int64_t seq, int64_t boundary, int sink, int tail, int packed) {
    for (int i = threadIdx.x; i < n64; i += 256) {
        const int t = i - 2;
        wide[i] = i == 0 ? (seq > 0 ? seq - 1 : 0) : i == 1 ? seq : t >= tail ? 0 : t < sink ? t : boundary + (t - sink);
    }
    if (threadIdx.x < 2) reinterpret_cast<int32_t*>(wide + n64)[threadIdx.x] = threadIdx.x ? tail : packed;
}

int step_block(int32_t* block, int n64, int64_t seq, int64_t boundary, int sink, int tail, int packed, void* stream) {
    if (n64 < 2 || tail < 0 || tail > n64 - 2) { set_error("step_block: bad shape"); return -1; }
    hipLaunchKernelGGL(step_block_kernel, dim3(1), dim3(256), 0, static_cast<hipStream_t>(stream), reinterpret_cast<int64_t*>(block), n64,
                       seq, boundary, sink, tail, packed);
    if (hipGetLastError() != hipSuccess) { set_error("step_block: launch failed"); return -2; }
    return 0;
}

// One workgroup per group of the list.
constexpr int kPackPairs = kUploadWords / 2;
__global__ void __launch_bounds__(128) pack_list_kernel(int32_t* src_rows, int32_t* dst_pages, int32_t* dst_groups,
                                                        int gt, int ppg, int hist_rows, int sink, int span,
                                                        int window_sink, int groups_per_seq, int pages_per_seq,
                                                        Words pairs) {
    const int n = blockIdx.x, r = pairs.w[2 * n], g = pairs.w[2 * n + 1], t = threadIdx.x;
    if (t < gt)
        src_rows[n * gt + t] = r * hist_rows + static_cast<int32_t>(ring_slot(window_sink + g * gt + t, sink, span));
    if (t < ppg) dst_pages[n * ppg + t] = r * pages_per_seq + g * ppg + t;
    if (t == 0) dst_groups[n] = r * groups_per_seq + g;
}

int pack_list(const int32_t* host_pairs, int n, int32_t* src_rows, int32_t* dst_pages, int32_t* dst_groups, int gt,
              int ppg, int hist_rows, int sink, int span, int window_sink, int groups_per_seq, int pages_per_seq,
              void* stream) {
    if (gt > 128 || ppg > gt) { set_error("pack_list: bad group size"); return -1; }
    Words w;
    for (int done = 0; done < n; done += kPackPairs) {
        const int m = n - done < kPackPairs ? n - done : kPackPairs;
        for (int i = 0; i < 2 * m; ++i) w.w[i] = host_pairs[2 * done + i];
        hipLaunchKernelGGL(pack_list_kernel, dim3(m), dim3(128), 0, static_cast<hipStream_t>(stream),
                           src_rows + done * gt, dst_pages + done * ppg, dst_groups + done, gt, ppg, hist_rows, sink,
                           span, window_sink, groups_per_seq, pages_per_seq, w);
    }
    if (hipGetLastError() != hipSuccess) { set_error("pack_list: launch failed"); return -2; }
    return 0;
}

}  // namespace ommx
