// Causal attention of prompt rows over their own bf16 K/V: the read side of a full-prefill step (the
// reference leaves it to the engine's varlen kernel, ommx_gpu_serve/integration/vllm/backend.py).
// Grouped-query heads, any number of requests per launch, head_dim 64 or 128.
//
// Precision is that of an fp32 softmax: q.k of bf16 operands is exact in the fp32 accumulator, the weights
// p = exp2(s - m) are fp32, and they enter P.V whole: p is cut into three bf16 pieces (8 + 8 + 8 bits,
// by truncation, so p = p0 + p1 + p2 exactly) that go through three matrix instructions against the
// same V operand.
//
// Layout.  A workgroup is four waves = 128 query rows of one q head; a wave owns 32 rows and walks the keys
// 64 at a time with mfma_f32_32x32x16_bf16.  Scores are formed transposed, S^T = K.Q^T, so a lane
// holds 32 scores of ONE query row: maximum and sum are register work plus one exchange with the
// other half of the wave.  The accumulator rows a lane holds (8j + 4*half + 0..3) are, in this order, what
// the B operand of O^T = V^T.P^T wants for a 16-key block once V^T lists its keys in the same order,
// so the weights never pass through LDS.  K rows and transposed V go to LDS, double buffered (64 KB,
// two workgroups per compute unit), 16-byte chunks XOR-swizzled by row: reads of eight rows hit eight
// different bank groups, and so do the transposing writes.  The next tile's rows are requested before a
// tile is worked on.
//
// Bound: matrix instructions, four units (one QK, three PV) where a bf16-weight kernel has two: 4096 tokens of
// 32 heads are 275 GFLOP issued, 0.11 ms at the card's peak rate.  The library's fp32 attention took
// 2.45 ms for them plus 0.1 ms of widening and repeating its inputs.
#include "ommx_common.h"
#include "ommx_internal.h"

namespace ommx {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

struct PrefillArgs {
    const uint16_t *q, *k, *v;
    int64_t q_t, q_h, k_t, k_h, v_t, v_h;
    float* o;
    uint16_t* o16;
    int64_t o_t, o_h;
    int Hkv, R;
    float scale_log2;            // softmax scale times log2(e)
};

constexpr int QROWS = 128, KEYS = 64;
// {first row of the request, its length, first query row of the tile within it}
constexpr int kTilesPerLaunch = kUploadWords / 3;
struct TileList { int32_t w[kUploadWords]; };

__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ float other_half(float v) { return __shfl_xor(v, 32); }
// high halves of two words: elements 0 and 1 of a packed bf16 pair, truncated
__device__ __forceinline__ uint32_t hi_pair(float lo, float hi) {
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}

// the running maximum is refreshed when a score (base 2) exceeds it by this: any bound that keeps
// exp2 in range serves an online softmax, and most tiles then rescale nothing
constexpr float MAX_SLACK = 8.0f;

template <int D>
__global__ void __launch_bounds__(256, 2) prefill_kernel(PrefillArgs a, TileList tiles) {
    constexpr int KB = D / 16;           // 16-channel blocks of QK
    constexpr int DB = D / 32;           // 32-channel blocks of the output
    constexpr int CHUNKS = D / 8;        // 16-byte chunks of a K row
    constexpr int K_BYTES = KEYS * D * 2, V_BYTES = D * KEYS * 2;
    constexpr int KLOADS = KEYS * CHUNKS / 256;
    extern __shared__ __attribute__((aligned(16))) uint8_t sm[];        // two buffers of K_BYTES + V_BYTES
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, half = lane >> 5;
    const int t0 = tiles.w[3 * blockIdx.y], len = tiles.w[3 * blockIdx.y + 1], q0 = tiles.w[3 * blockIdx.y + 2];
    // (neighbouring workgroups take neighbouring kv heads, so with 8 kv heads an XCD keeps to one)
    const int kvh = blockIdx.x % a.Hkv, h = kvh * a.R + blockIdx.x / a.Hkv;
    const uint16_t* const kp = a.k + t0 * a.k_t + kvh * a.k_h;
    const uint16_t* const vp = a.v + t0 * a.v_t + kvh * a.v_h;

    const int row_first = q0 + 32 * wave, row = row_first + col;         // of this wave, of this lane
    u32x4 qf[KB];
    {
        const uint16_t* qp = a.q + (t0 + min(row, len - 1)) * a.q_t + h * a.q_h + 8 * half;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) qf[kb] = *reinterpret_cast<const u32x4*>(qp + 16 * kb);
    }
    f32x16 acc[DB];
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[d][r] = 0.0f;
    float m = -INFINITY, l = 0.0f;

    const int n_tiles = (min(len, q0 + QROWS) + KEYS - 1) / KEYS;

    // ---- staging: thread -> chunk tid % CHUNKS of K rows, and channels 8*d8.. of four neighbouring V rows
    const int kc = tid % CHUNKS, kr = tid / CHUNKS;
    const int d8 = tid % CHUNKS, kg = tid / CHUNKS;
    constexpr int VGROUPS = KEYS / 4;                       // groups of four keys
    const bool v_mine = kg < VGROUPS;                       // head_dim 64: half of the threads
    u32x4 kn[KLOADS], vn[4];
    auto request = [&](int k0) {
#pragma unroll
        for (int i = 0; i < KLOADS; ++i) {
            const int key = min(k0 + kr + i * (256 / CHUNKS), len - 1);
            kn[i] = *reinterpret_cast<const u32x4*>(kp + key * a.k_t + 8 * kc);
        }
        if (v_mine) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = min(k0 + 4 * kg + i, len - 1);
                vn[i] = *reinterpret_cast<const u32x4*>(vp + key * a.v_t + 8 * d8);
            }
        }
    };
    auto stage = [&](uint8_t* buf) {
#pragma unroll
        for (int i = 0; i < KLOADS; ++i) {
            const int r = kr + i * (256 / CHUNKS);
            *reinterpret_cast<u32x4*>(buf + r * (2 * D) + 16 * (kc ^ (r & 7))) = kn[i];
        }
        if (v_mine) {
            // keys 4kg..4kg+3 are block kg / 4, half kg & 1 of it, first or second four slots of that chunk
            const int chunk = 2 * (kg >> 2) + (kg & 1), part = (kg >> 1) & 1;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
#pragma unroll
                for (int odd = 0; odd < 2; ++odd) {
                    const uint32_t sel = odd ? 0x07060302u : 0x05040100u;
                    const u32x2 four = {__builtin_amdgcn_perm(vn[1][w], vn[0][w], sel),
                                        __builtin_amdgcn_perm(vn[3][w], vn[2][w], sel)};
                    const int d = 8 * d8 + 2 * w + odd;
                    *reinterpret_cast<u32x2*>(buf + K_BYTES + d * (2 * KEYS) + 16 * (chunk ^ (d & 7) ^ (d8 & 7)) + 8 * part) = four;
                }
            }
        }
    };

    request(0);
    stage(sm);
    __syncthreads();
    for (int t = 0; t < n_tiles; ++t) {
        const int k0 = t * KEYS;
        uint8_t* const buf = sm + (t & 1) * (K_BYTES + V_BYTES);
        if (t + 1 < n_tiles) request(k0 + KEYS);
        if (row_first < len && k0 <= row_first + 31) {
            // ---------------------------------------------------------------- S^T = K.Q^T
            f32x16 s[2];
#pragma unroll
            for (int g = 0; g < 2; ++g) {
#pragma unroll
                for (int r = 0; r < 16; ++r) s[g][r] = 0.0f;
                const int key = 32 * g + col;
#pragma unroll
                for (int kb = 0; kb < KB; ++kb) {
                    const u32x4 kf = *reinterpret_cast<const u32x4*>(buf + key * (2 * D) + 16 * ((2 * kb + half) ^ (key & 7)));
                    s[g] = mfma32(kf, qf[kb], s[g]);
                }
            }
            // ---------------------------------------------------------------- online softmax of one row
            if (k0 + KEYS - 1 > row_first) {
#pragma unroll
                for (int g = 0; g < 2; ++g)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if (k0 + 32 * g + 8 * (r >> 2) + 4 * half + (r & 3) > row) s[g][r] = -INFINITY;
            }
            float mx = s[0][0];
#pragma unroll
            for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[0][r]);
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[1][r]);
            mx = fmaxf(mx, other_half(mx)) * a.scale_log2;      // (the scale is positive)
            if (__any(mx > m + MAX_SLACK)) {
                const float m_new = fmaxf(m, mx);
                const float shrink = __builtin_amdgcn_exp2f(m - m_new);       // 0 on the first tile
                m = m_new;
                l *= shrink;
#pragma unroll
                for (int d = 0; d < DB; ++d)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[d][r] *= shrink;
            }
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    s[g][r] = __builtin_amdgcn_exp2f(fmaf(s[g][r], a.scale_log2, -m));
                    l += s[g][r];
                }
            // ---------------------------------------------------------------- O^T += V^T.P^T
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                u32x4 p0, p1, p2;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float x = s[b >> 1][8 * (b & 1) + 2 * i], y = s[b >> 1][8 * (b & 1) + 2 * i + 1];
                    const float x1 = x - __uint_as_float(__float_as_uint(x) & 0xFFFF0000u);
                    const float y1 = y - __uint_as_float(__float_as_uint(y) & 0xFFFF0000u);
                    const float x2 = x1 - __uint_as_float(__float_as_uint(x1) & 0xFFFF0000u);
                    const float y2 = y1 - __uint_as_float(__float_as_uint(y1) & 0xFFFF0000u);
                    p0[i] = hi_pair(x, y);
                    p1[i] = hi_pair(x1, y1);
                    p2[i] = hi_pair(x2, y2);
                }
#pragma unroll
                for (int d = 0; d < DB; ++d) {
                    const int ch = 32 * d + col;
                    const u32x4 vf = *reinterpret_cast<const u32x4*>(
                        buf + K_BYTES + ch * (2 * KEYS) + 16 * ((2 * b + half) ^ (ch & 7) ^ ((ch >> 3) & 7)));
                    acc[d] = mfma32(vf, p0, acc[d]);
                    acc[d] = mfma32(vf, p1, acc[d]);
                    acc[d] = mfma32(vf, p2, acc[d]);
                }
            }
        }
        if (t + 1 < n_tiles) stage(sm + ((t + 1) & 1) * (K_BYTES + V_BYTES));
        __syncthreads();
    }

    if (row >= len) return;
    l += other_half(l);
    const float inv = 1.0f / l;
    const int64_t at = (t0 + row) * a.o_t + h * a.o_h;
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            const int ch = 32 * d + 8 * r4 + 4 * half;
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = acc[d][4 * r4 + i] * inv;
            if (a.o16)
                *reinterpret_cast<u32x2*>(a.o16 + at + ch) =
                    u32x2{f32_to_bf16_any(v[0]) | (static_cast<uint32_t>(f32_to_bf16_any(v[1])) << 16),
                          f32_to_bf16_any(v[2]) | (static_cast<uint32_t>(f32_to_bf16_any(v[3])) << 16)};
            else
                *reinterpret_cast<float4*>(a.o + at + ch) = float4{v[0], v[1], v[2], v[3]};
        }
}

template <int D>
void launch(const PrefillArgs& a, const TileList& list, int n, hipStream_t st) {
    const size_t shm = 2 * (2 * KEYS * D * 2);
    hipLaunchKernelGGL((prefill_kernel<D>), dim3(a.Hkv * a.R, n), dim3(256), shm, st, a, list);
}

}  // namespace

int prefill_attention(const uint16_t* q, int64_t q_t, int64_t q_h, const uint16_t* k, int64_t k_t, int64_t k_h,
                      const uint16_t* v, int64_t v_t, int64_t v_h, void* o, bool o_bf16, int64_t o_t, int64_t o_h,
                      const int64_t* host_starts, int B, int Hq, int Hkv, int D, float scale, void* stream) {
    const char* bad = nullptr;
    if (B < 1 || Hkv < 1 || Hq % Hkv || !(D == 64 || D == 128) || !(scale > 0.0f)) bad = "prefill_attention: bad shape";
    else if (((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) |
               reinterpret_cast<uintptr_t>(o)) & 15) ||
             (q_t | q_h | k_t | k_h | v_t | v_h | o_t | o_h) % 8)
        bad = "prefill_attention: rows must be 16-byte aligned";
    if (bad) { set_error(bad); return -1; }
    const PrefillArgs a{q, k, v, q_t, q_h, k_t, k_h, v_t, v_h, o_bf16 ? nullptr : static_cast<float*>(o),
                        o_bf16 ? static_cast<uint16_t*>(o) : nullptr, o_t, o_h, Hkv, Hq / Hkv,
                        scale * 1.4426950408889634f};
    // Tiles of 128 query rows, those with the most keys first: the grid drains evenly.
    int most = 0;
    for (int b = 0; b < B; ++b) {
        const int64_t n = host_starts[b + 1] - host_starts[b];
        if (n > most) most = static_cast<int>(n);
    }
    TileList list;
    int n = 0;
    hipStream_t st = static_cast<hipStream_t>(stream);
    auto flush = [&]() {
        if (n == 0) return;
        if (D == 128) launch<128>(a, list, n, st); else launch<64>(a, list, n, st);
        n = 0;
    };
    for (int q0 = (most - 1) / QROWS * QROWS; q0 >= 0; q0 -= QROWS)
        for (int b = 0; b < B; ++b) {
            const int len = static_cast<int>(host_starts[b + 1] - host_starts[b]);
            if (q0 >= len) continue;
            list.w[3 * n] = static_cast<int32_t>(host_starts[b]);
            list.w[3 * n + 1] = len;
            list.w[3 * n + 2] = q0;
            if (++n == kTilesPerLaunch) flush();
        }
    flush();
    if (hipGetLastError() != hipSuccess) { set_error("prefill_attention: launch failed"); return -2; }
    return 0;
}

}  // namespace ommx
