// gemm_split.hpp -- FP32 activations as pairs of fp16 values, the A operand of
// the expert GEMMs (expert_gemm.hip).
//
// A row (or a 32-value chunk of a row) gets a power-of-two scale s that brings
// its largest magnitude into [2^14, 2^15); then x / s = hi + lo with hi = the
// fp16 nearest x / s and lo = the fp16 nearest the rest.  hi + lo keeps 22 to 23
// significant bits of every value above 2^-15 of the row's maximum and an
// absolute error of 2^-39 of that maximum below (fp16 subnormals, which the
// MFMA reads exactly): FP32's own rounding, at two MFMAs per product where
// three bf16 parts take three.  Chunks are brought to their row's scale by a power
// of two when the GEMM loads them, which rounds their halves to the same absolute
// step: 2^-38 of the row's maximum at most.
//
// Rows are stored as [row][32-value stage][hi, lo][32], so one stage of a row
// is one 128-byte line; inside each run of 8 values the order is 0, 2, 1, 3, 4,
// 6, 5, 7, the order in which masking 4-bit or 8-bit weight fields out of a dword
// leaves them (kPairOrder).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pk {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// Position of value e (0..7) of a run of 8 in the stored order (its own inverse).
__device__ __forceinline__ constexpr uint32_t kPairOrder(uint32_t e) {
    return (e & 4u) | ((e & 1u) << 1) | ((e >> 1) & 1u);
}

// The scale of a row or chunk of maximum magnitude m, and its inverse (both
// powers of two; an infinite or NaN maximum gives finite scales and a row that
// stays non-finite; a zero row gets the smallest scale).
__device__ __forceinline__ void split_scale(float m, float& s, float& inv) {
    uint32_t e = (__float_as_uint(m) >> 23) & 0xffu;
    e = e < 15u ? 15u : e;
    s = __uint_as_float((e - 14u) << 23);
    inv = __uint_as_float((268u - e) << 23);
}

constexpr float kZeroScale = 0x1p-126f;  // the scale of a zero row or chunk (or one below 2^-112)

// Two scaled values as (hi, hi) and (lo, lo) dwords.
__device__ __forceinline__ void split_pair(float a, float b, uint32_t& hi, uint32_t& lo) {
    const f16x2 h = {static_cast<_Float16>(a), static_cast<_Float16>(b)};
    const float ra = a - static_cast<float>(h.x), rb = b - static_cast<float>(h.y);
    const f16x2 l = {static_cast<_Float16>(ra), static_cast<_Float16>(rb)};
    hi = __builtin_bit_cast(uint32_t, h);
    lo = __builtin_bit_cast(uint32_t, l);
}

}  // namespace pk
