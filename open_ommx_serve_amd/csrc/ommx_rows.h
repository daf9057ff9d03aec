// Rows of a prompt block on their way into the bf16 row history (csrc/ommx_ring.hip describes the ring): a workgroup copies
// one row of H*D elements, K and V, eight elements (16 bytes of bf16) per thread and turn.
#pragma once
#include "ommx_common.h"
#include "ommx_internal.h"

namespace ommx {

__device__ __forceinline__ int64_t ring_slot(int64_t pos, int sink, int span) {
    if (span <= 0 || pos < sink) return pos;
    const int64_t past = pos - sink;
    if (past >> 32 == 0) return sink + static_cast<uint32_t>(past) % static_cast<uint32_t>(span);    // a third of the steps
    return sink + past % span;
}

template <bool F32>
__device__ __forceinline__ void put8(uint16_t* dst, const void* src, int64_t at, bool vec) {
    if constexpr (F32) {
        const float* p = static_cast<const float*>(src) + at;
#pragma unroll
        for (int i = 0; i < 8; ++i) dst[i] = f32_to_bf16_any(p[i]);
    } else {
        const uint16_t* p = static_cast<const uint16_t*>(src) + at;
        if (vec) *reinterpret_cast<uint4*>(dst) = *reinterpret_cast<const uint4*>(p);
        else
#pragma unroll
            for (int i = 0; i < 8; ++i) dst[i] = p[i];
    }
}

// MAY_F32: the source may be fp32 (rounded as torch does)
template <bool MAY_F32>
__device__ __forceinline__ void copy_block_row(const BlockRows& a, int n) {
    const int row = n < a.n_head ? n : a.lo + (n - a.n_head);
    const int64_t at = ring_slot(a.pos0 + row, a.sink, a.span) * static_cast<int64_t>(a.H * a.D);
    const int per_head = a.D / 8;
    for (int i = threadIdx.x; i < a.H * per_head; i += blockDim.x) {
        const int h = i / per_head, c = (i % per_head) * 8;
        const int64_t k_at = row * a.k_ts + h * a.k_hs + c, v_at = row * a.v_ts + h * a.v_hs + c;
        const int64_t to = at + h * a.D + c;
        if (MAY_F32 && a.k_f32) put8<true>(a.k_hist + to, a.K, k_at, false); else put8<false>(a.k_hist + to, a.K, k_at, a.k_vec);
        if (MAY_F32 && a.v_f32) put8<true>(a.v_hist + to, a.V, v_at, false); else put8<false>(a.v_hist + to, a.V, v_at, a.v_vec);
    }
}

// Row b of a step to its place, and the step's numbers of request b to the block that its other launches read, as ring_step_kernel
// (ommx_ring.hip) does.
template <int D>
__device__ __forceinline__ void copy_step_row(const StepWrite& s, int b) {
    const int p = s.at.pos[b], slot = s.at.slot[b], B = s.B;
    if (s.block && threadIdx.x == 0) {
        int64_t* const wide = reinterpret_cast<int64_t*>(s.block);
        wide[b] = slot;
        wide[B + b] = p;
        wide[2 * B + b] = p + 1LL;
        s.block[6 * B + b] = s.at.packed[b];
    }
    const int64_t row = ring_slot(p, s.sink, s.span);
    if (row < 0 || row >= s.rows) {
        if (s.err && threadIdx.x == 0) atomicOr(s.err, OMMX_ERR_RING_RANGE);
        return;
    }
    const int64_t to = slot * s.stride_req + row * static_cast<int64_t>(s.H * D);
    for (int i = threadIdx.x; i < s.H * (D / 8); i += blockDim.x) {
        const int h = i / (D / 8), c = 8 * (i % (D / 8));
        const uint4 x = *reinterpret_cast<const uint4*>(s.k + b * s.k_bs + h * s.k_hs + c);
        const uint4 y = *reinterpret_cast<const uint4*>(s.v + b * s.v_bs + h * s.v_hs + c);
        *reinterpret_cast<uint4*>(s.k_hist + to + h * D + c) = x;
        *reinterpret_cast<uint4*>(s.v_hist + to + h * D + c) = y;
    }
}

}  // namespace ommx
