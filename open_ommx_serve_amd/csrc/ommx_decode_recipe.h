// Limits and small helpers of the serving-recipe decode kernels (ommx_decode_gqa4.hip, ommx_decode_team.hip).
#pragma once
#include "ommx_decode_util.h"

namespace ommx {
namespace decode_util {

// One f16 carries 11 bits: rounding an outlier delta d costs up to |d| * 2^-11, i.e. up to
// |d| * max|q| * 2^-11 * sm_scale on a logit.  A delta with |d| * max|q| >= BIG_DELTA * 16
// (at most 1.4e-3 on a logit at sm_scale = 128^-0.5) gets its residual added exactly; smaller
// ones stay below that and average a quarter of it.  The bound is held at other sm_scale values
// (head_dim 64: 64^-0.5) by dividing the threshold by sm_scale / 128^-0.5; the general form, with
// up to 8 entries per vector, takes three quarters of it, and half with fewer than 6 outlier slots (more
// large values then stay in the base codes, the steps grow, and so do the entries).
constexpr float BIG_DELTA = 2.0f;
constexpr float BIG_DELTA_SM_SCALE = 0.08838834764831845f;
// The base operand (1 + code*2^(2m-10)) * 2^e carries a constant A*2^e per channel, up to 2^6 times
// the signal, which the bias MFMA takes out again: two large sums that cancel in fp32.  From steps
// of 2^EXACT_STEP_EXP on (values a hundred or more wide inside one vector) that shows on the logits, and
// the step's two groups take the operand code*2^(2m-10+e) instead (one packed subtraction more per operand
// register, exact: both terms share the exponent) and drops the 2^e bias column.
constexpr int EXACT_STEP_EXP = 5;
// f16 operands: steps above 2^15 do not fit (K or V values beyond some 1e5); such a step is held at 2^15
// and OMMX_ERR_VALUE_RANGE is reported
constexpr int MAX_STEP_EXP = 15;
// largest step whose 2^24-fold over the smallest A scale, 4, is an fp32 number
constexpr int CODE_STEP_EXP = 105;

// Outlier positions of a bitmap from below: the lowest set bit (-1 of an empty map, see LdsMap), and the map without the bit at
// `pos`, one addition of -1 << pos (m & (m - 1) takes two instructions).
__device__ __forceinline__ int lowest_bit(uint32_t m) {
    int pos;
    asm("v_ffbl_b32 %0, %1" : "=v"(pos) : "v"(m));
    return pos;
}
__device__ __forceinline__ uint32_t without_bit(uint32_t m, int pos) {
    uint32_t r;
    asm("v_lshl_add_u32 %0, -1, %1, %2" : "=v"(r) : "v"(pos), "v"(m));
    return r;
}
__device__ __forceinline__ float f16_bits(uint32_t b) { return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(b))); }

}  // namespace decode_util
}  // namespace ommx
