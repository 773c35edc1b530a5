// expert_gemm.hip -- the grouped expert GEMMs of the batched prefill, on fp16 MFMA.
//
// Per tile of 64 (or, for an expert's last rows, 32) assignments and 256 weight
// rows: the weights' integer fields go from memory straight into the registers
// of the wave that uses them and become fp16 operands by masking alone; the
// activations, split into two fp16 values each (gemm_split.hpp), pass through
// LDS, shared by the four waves.  Both products of a weight with an
// activation's two halves are exact in the FP32 accumulator.
//
// What bounds it: the vector ALU beside the MFMAs (weight fields to operands,
// scale groups into the accumulators) and the waits between them.  So a decoded
// weight serves two 32-row blocks, two fp16 halves replace three bf16 parts,
// Q4_K's scales go into the integers instead of one FMA per element and group,
// and the K order inside a group is the one the masks leave.  Against 32-row
// tiles of three bf16 parts with 128-biased weights, hidden 2048, ffn 768, 128
// experts, top-8, Q4_K / Q6_K: 4096 tokens gate/up 918 -> 472 us, down 636 ->
// 403 us; 512 tokens (skewed load) 193 -> 118 and 141 -> 103 us.  (Loads of weights
// as whole lines through LDS, fragments read half a step ahead with a barrier
// every second step, and both: the same gate/up time, slower down.)  Error against
// float64 on the same inputs, before and after: Q4_K/Q6_K 3.8e-6 -> 7.8e-7,
// Q6_K 9.7e-7 -> 3.6e-7, Q5_K 4.4e-7 -> 3.7e-7, Q8_0 4.4e-7 -> 3.0e-7, Q4_0
// 4.4e-7 -> 2.9e-7, Q4_1 4.6e-7 -> 4.0e-7.
#include <math.h>

#include "gemm_split.hpp"
#include "kquant.hpp"
#include "launch.hpp"
#include "route.hpp"

namespace pk {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16 mfma(f16x8 a, f16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f16x8 frag4(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_bit_cast(f16x8, make_uint4(a, b, c, d));
}
__device__ __forceinline__ uint32_t pk_add16(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, a) + __builtin_bit_cast(f16x2, b));
}
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pk_mul_u16(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, static_cast<u16x2>(__builtin_bit_cast(u16x2, a) *
                                                           __builtin_bit_cast(u16x2, b)));
}
__device__ __forceinline__ uint32_t pk_fma16(uint32_t a, f16x2 b, uint32_t c) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(f16x2, a), b,
                                                                  __builtin_bit_cast(f16x2, c)));
}
__device__ __forceinline__ uint32_t pk_mul_f16(uint32_t a, f16x2 b) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, a) * b);
}

// ---------------------------------------------------------------------------
// Weights as fp16 operands, 256 values (a superblock) of one row per lane pair.
//
// Lane (n = lane % 32, kq = lane / 32) feeds row n.  Step j of a superblock is
// its 32-value group j, two B fragments of 8 values per lane: values 16 kq + 8 h
// .. + 7 of the group (kHalfRuns: a lane reads 16 consecutive quant bytes) or
// 16 h + 8 kq .. + 7, for fragment h; the A fragments follow (frag_piece).
//
// Q4_K, Q5_K (kSuper): the group's 6-bit scale times the 4- or 5-bit quant is an
// integer below 2^11, whose bits are the fp16 value 2^-24 times it (subnormals
// and the first binade are linear), so a masked pair times the scale pair
// (v_pk_mul_lo_u16) is the operand and only d and the mins are left outside.
//  * Q4_K in the MoE block (kUnits): the accumulator is kept in units of the superblock's d and
//    rescaled by d_prev / d once per 256 values.  The mins' term is one more
//    MFMA per superblock: the eight integer mins against the eight group sums of
//    x (split hi and lo, 16 operand values).
//  * Q5_K, and Q4_K in the prompt's projections: q - 16 (q - 8), the rest of the mins'
//    term (16 d sc - dmin m) times the FP32 group sums on FP32 MFMA.  With two row
//    blocks each step's sum goes into the accumulator by an FMA with d, as the other
//    formats' do; with one there are registers for sums over the superblock (kSums),
//    as the FMA per step would wait for its products there (77 tokens, hidden 1024,
//    prefill 69.9 -> 74.8 us).  Q5_K keeps the high and the low halves' apart: a single sum
//    was 20% further from float64 at hidden 512 (3.5e-7 against 2.9e-7; 1024: 3.7e-7
//    against 3.2e-7, 2048: 4.5e-7 against 4.3e-7), and with two row blocks spilled 13 to
//    23 registers (2048 tokens 735 -> 701 us without, 77 tokens 68.7 -> 69.4).  Only at
//    hidden 4096 and two row blocks, where the FMAs are many, was it closer (4.7e-7
//    against 5.0e-7; exact bf16 parts 5.6e-7); two steps to an FMA spill again.  Q4_K
//    projections keep the single sum (4.0e-7): the model's logits are as far from
//    float64 as with a token step per position (0.995 +- 0.014 of that over 294 prompts).
//    As kUnits, Q5_K had 6.1e-7 (the larger quants leave more to cancel against the
//    mins), and Q4_K projections at 8.7e-7 put the whole model's logits 15% further from
//    float64, as fewer FP16 roundings of k then agree; the MoE block's gate/up keeps the
//    units, 472 against 557 us at 4096 tokens, and does not show in the logits.
//
// The others: quants as exact fp16 integers around zero (1024 + q by or-ing the
// exponent in, minus 1024 and the offset), and per scale group (32 values;
// Q6_K 16) acc += ds * P.  Q4_1's m + 8 d goes in as Q5_K's mins do.
// (Small integers as subnormal codes would lose bits: the MFMA aligns them as if
// their top bit were set.)

template <int T, bool UNITS>
struct WTraits {
    static constexpr bool kSuper = T == T_Q4_K || T == T_Q5_K;
    static constexpr bool kMins = kSuper || T == T_Q4_1;
    static constexpr bool kUnits = T == T_Q4_K && UNITS;           // accumulator in units of d
    static constexpr bool kMinsF32 = kMins && !kUnits;    // mins' term on FP32 MFMA
    static constexpr bool kHalfRuns = kSuper || T == T_Q8_0;
    static constexpr uint32_t kGroup = T == T_Q6_K ? 16u : 32u;
};

template <int T> struct WRaw;  // a lane's fields of one row, loaded ahead
template <> struct WRaw<T_Q4_K> { uint32_t q[4][4]; uint32_t h[4]; };
template <> struct WRaw<T_Q5_K> { uint32_t q[4][4]; uint32_t h[4]; uint32_t qh[4]; };
template <> struct WRaw<T_Q6_K> { uint32_t ql[2][2][4]; uint32_t qh[2][4]; uint32_t sc[4]; uint32_t d; };
template <> struct WRaw<T_Q8_0> { uint32_t q[4][4]; uint32_t d[4]; };   // ring of four steps
template <> struct WRaw<T_Q4_0> { uint32_t q[8][2]; uint32_t d[4]; };
template <> struct WRaw<T_Q4_1> { uint32_t q[4][2]; uint32_t dm[4]; };  // ring of four steps

// What a superblock's steps share, taken from the header fields at its start
// (which then reload for the next superblock).
template <int T> struct WHead;
template <> struct WHead<T_Q4_K> { uint32_t sc[2]; float cn[4]; float d; };
template <> struct WHead<T_Q5_K> { uint32_t sc[2]; uint32_t qh[4]; float cn[4]; float d; };
template <> struct WHead<T_Q6_K> { uint32_t sc[4]; float d; };
template <> struct WHead<T_Q8_0> { uint32_t d[4]; };
template <> struct WHead<T_Q4_0> { uint32_t d[4]; };
template <> struct WHead<T_Q4_1> { float cn[4]; };

// Where a lane's row lies: per plane a uniform base of the workgroup's first
// row (32-bit lane offsets from it).
template <int T>
struct WSrc {
    const uint8_t* p0;  // GGUF form: the blocks; planar: the largest plane
    const uint8_t* p1;
    const uint8_t* p2;
    const uint8_t* p3;
};

// Planes of rows starting at block blk0 of a slice of nblk blocks.
template <int T>
__device__ __forceinline__ WSrc<T> wsrc(const uint8_t* slice, uint64_t nblk, uint64_t blk0) {
    WSrc<T> s;
    s.p1 = s.p2 = s.p3 = nullptr;
    if constexpr (T == T_Q6_K) {
        using L = Planar<T_Q6_K>;
        s.p0 = slice + nblk * L::QL + blk0 * 128u;
        s.p1 = slice + nblk * L::QH + blk0 * 64u;
        s.p2 = slice + nblk * L::SC + blk0 * 16u;
        s.p3 = slice + nblk * L::D + blk0 * 2u;
    } else if constexpr (T == T_Q8_0) {
        using L = Planar<T_Q8_0>;
        s.p0 = slice + nblk * L::QS + blk0 * 32u;
        s.p1 = slice + nblk * L::D + blk0 * 2u;
    } else if constexpr (T == T_Q4_0) {
        using L = Planar<T_Q4_0>;
        s.p0 = slice + nblk * L::QS + blk0 * 16u;
        s.p1 = slice + nblk * L::D + blk0 * 2u;
    } else {
        s.p0 = slice + blk0 * Fmt<T>::BB;
    }
    return s;
}

__device__ __forceinline__ void ld4(const uint8_t* p, uint32_t (&w)[4]) { ld_words<4>(p, w); }
__device__ __forceinline__ void ld2(const uint8_t* p, uint32_t (&w)[2]) { ld_words<2>(p, w); }

// Header fields of superblock b (blk: the lane's row's first block, relative
// to the source's base).
template <int T>
__device__ __forceinline__ void wload_head(const WSrc<T>& s, uint32_t blk, uint32_t b, uint32_t kq,
                                           WRaw<T>& r) {
    if constexpr (T == T_Q4_K) {
        ld4(s.p0 + (blk + b) * 144u, r.h);
    } else if constexpr (T == T_Q5_K) {
        ld4(s.p0 + (blk + b) * 176u, r.h);
        ld4(s.p0 + (blk + b) * 176u + 16u + 16u * kq, r.qh);
    } else if constexpr (T == T_Q6_K) {
        ld4(s.p2 + (blk + b) * 16u, r.sc);
        r.d = ld_u16(s.p3 + (blk + b) * 2u);
    } else if constexpr (T == T_Q8_0 || T == T_Q4_0) {
        ld4(s.p1 + (blk + 8u * b) * 2u, r.d);
    }
}

// Quants that step j of superblock b starts with (nothing where an earlier
// step's load covers it).  The lane's offset of the superblock stands apart from
// the step's constant one, which goes into the load instruction.
template <int T>
__device__ __forceinline__ void wload_step(const WSrc<T>& s, uint32_t blk, uint32_t b, uint32_t j,
                                           uint32_t kq, WRaw<T>& r) {
    if constexpr (T == T_Q4_K || T == T_Q5_K) {
        const uint8_t* p = s.p0 + ((blk + b) * Fmt<T>::BB + 16u * kq);
        if (j % 2u == 0u) ld4(p + (T == T_Q4_K ? 16u : 48u) + 16u * j, r.q[j / 2u]);
    } else if constexpr (T == T_Q6_K) {
        // half hh of the block: two ql runs (steps 4 hh + 0, 2 and + 1, 3), one qh run
        const uint32_t hh = j / 4u, g = j % 4u;
        const uint8_t* p = s.p0 + ((blk + b) * 128u + 16u * kq);
        const uint8_t* ph = s.p1 + ((blk + b) * 64u + 16u * kq);
        if (g < 2u) ld4(p + 64u * hh + 32u * g, r.ql[hh][g]);
        if (g == 0u) ld4(ph + 32u * hh, r.qh[hh]);
    } else if constexpr (T == T_Q8_0) {
        const uint8_t* p = s.p0 + ((blk + 8u * b) * 32u + 16u * kq);
        ld4(p + 32u * j, r.q[j % 4u]);
    } else if constexpr (T == T_Q4_0) {
        const uint8_t* p = s.p0 + ((blk + 8u * b) * 16u + 8u * kq);
        ld2(p + 16u * j, r.q[j]);
    } else if constexpr (T == T_Q4_1) {
        const uint8_t* p = s.p0 + (blk + 8u * b) * 20u;
        const uint8_t* pq = s.p0 + ((blk + 8u * b) * 20u + 8u * kq);
        r.dm[j % 4u] = *reinterpret_cast<const uint32_t*>(__builtin_assume_aligned(p + 20u * j, 4));
        ld2(pq + 20u * j + 4u, r.q[j % 4u]);
    }
}

// The loads that refill what step j of superblock b has just consumed (`bn`:
// the superblock after b, clamped to the row's last).
template <int T>
__device__ __forceinline__ void wreload(const WSrc<T>& s, uint32_t blk, uint32_t b, uint32_t bn,
                                        uint32_t j, uint32_t kq, WRaw<T>& r) {
    if constexpr (T == T_Q4_K || T == T_Q5_K) {
        if (j % 2u == 1u) wload_step<T>(s, blk, bn, j - 1u, kq, r);
    } else if constexpr (T == T_Q6_K) {
        const uint32_t hh = j / 4u, g = j % 4u;
        const uint8_t* p = s.p0 + ((blk + bn) * 128u + 16u * kq);
        const uint8_t* ph = s.p1 + ((blk + bn) * 64u + 16u * kq);
        if (g >= 2u) ld4(p + 64u * hh + 32u * (g - 2u), r.ql[hh][g - 2u]);
        if (g == 3u) ld4(ph + 32u * hh, r.qh[hh]);
    } else if constexpr (T == T_Q8_0 || T == T_Q4_1) {
        if (j < 4u) wload_step<T>(s, blk, b, j + 4u, kq, r);
        else wload_step<T>(s, blk, bn, j - 4u, kq, r);
    } else {
        wload_step<T>(s, blk, bn, j, kq, r);
    }
}

// A 32-byte run loaded as lane kq's bytes 16 kq .. + 15: bytes 8 kq .. + 7 and
// 16 + 8 kq .. + 7 (the two lanes of a row trade the middle 8 bytes).
__device__ __forceinline__ void run_words(const uint32_t* w, uint32_t (&o)[4]) {
    const auto s02 = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
    const auto s13 = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
    o[0] = s02[0];
    o[1] = s13[0];
    o[2] = s02[1];
    o[3] = s13[1];
}

// The bytes of w as the fp16 pairs (0, 2) and (1, 3) of 1024 + byte.
__device__ __forceinline__ void bytes_1024(uint32_t w, uint32_t& even, uint32_t& odd) {
    even = __builtin_amdgcn_perm(0x64646464u, w, 0x04020400u);
    odd = __builtin_amdgcn_perm(0x64646464u, w, 0x04030401u);
}

__device__ __forceinline__ float half_of(const uint32_t* w, uint32_t i) {
    return half_bits_to_float((w[i / 2u] >> (16u * (i & 1u))) & 0xffffu);
}

constexpr uint32_t h16x2(uint32_t bits) { return bits | (bits << 16); }

// Step j's two B fragments, and (no kSuper) the scale of each.
template <int T, bool UNITS>
__device__ __forceinline__ void wfrag(const WRaw<T>& r, const WHead<T>& hd, uint32_t j, f16x8 (&b)[2],
                                      float (&ds)[2]) {
    uint32_t w[8];
    if constexpr (T == T_Q4_K || T == T_Q5_K) {
        const uint32_t c = j / 2u, hi = j & 1u;
        // byte j % 4 of the scale word, in both halves
        const f16x2 k4096 = {static_cast<_Float16>(4096.0f), static_cast<_Float16>(4096.0f)};
        uint32_t mid = 0u;  // set below: -16 sc 2^-12
        const uint32_t scp = __builtin_amdgcn_perm(0u, hd.sc[j / 4u], 0x0c000c00u + 0x00010001u * (j % 4u));
        if constexpr (!WTraits<T, UNITS>::kUnits) mid = pk_mul_f16((scp << (T == T_Q5_K ? 4 : 3)) | 0x80008000u, k4096);
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            uint32_t e, o;
            if constexpr (T == T_Q4_K) {
                const uint32_t q = r.q[c][i];
                e = (hi ? q >> 4 : q) & 0x000f000fu;
                o = (hi ? q >> 12 : q >> 8) & 0x000f000fu;
            } else {
                const uint32_t q = (hi ? r.q[c][i] >> 4 : r.q[c][i]) & 0x0f0f0f0fu;
                const uint32_t v = q | (((hd.qh[i] >> j) & 0x01010101u) << 4);
                e = v & 0x00ff00ffu;
                o = (v >> 8) & 0x00ff00ffu;
            }
            w[2u * i] = pk_mul_u16(e, scp);
            w[2u * i + 1u] = pk_mul_u16(o, scp);
            if constexpr (!WTraits<T, UNITS>::kUnits) {  // sc (q - 16) 2^-12: normal values, exact
                w[2u * i] = pk_fma16(w[2u * i], k4096, mid);
                w[2u * i + 1u] = pk_fma16(w[2u * i + 1u], k4096, mid);
            }
        }
        if constexpr (!WTraits<T, UNITS>::kUnits) ds[0] = ds[1] = hd.d;
    } else if constexpr (T == T_Q6_K) {
        const uint32_t hh = j / 4u, g = j % 4u;
        uint32_t ql[4], qh[4];
        run_words(r.ql[hh][g & 1u], ql);
        run_words(r.qh[hh], qh);
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            const uint32_t nib = (g >= 2u ? ql[i] >> 4 : ql[i]) & 0x0f0f0f0fu;
            uint32_t e, o;
            bytes_1024(nib | (((qh[i] >> (2u * g)) & 0x03030303u) << 4), e, o);
            w[2u * i] = pk_add16(e, h16x2(0xe420u));  // - 1056
            w[2u * i + 1u] = pk_add16(o, h16x2(0xe420u));
        }
        const uint32_t s2 = hd.sc[j / 2u] >> (16u * (j & 1u));
        ds[0] = __fmul_rn(hd.d, static_cast<float>(static_cast<int8_t>(s2 & 0xffu)));
        ds[1] = __fmul_rn(hd.d, static_cast<float>(static_cast<int8_t>((s2 >> 8) & 0xffu)));
    } else if constexpr (T == T_Q8_0) {
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            uint32_t e, o;
            bytes_1024(r.q[j % 4u][i] ^ 0x80808080u, e, o);
            w[2u * i] = pk_add16(e, h16x2(0xe480u));  // - 1152
            w[2u * i + 1u] = pk_add16(o, h16x2(0xe480u));
        }
        ds[0] = ds[1] = half_of(hd.d, j);
    } else {  // Q4_0, Q4_1: low nibbles are values 0..15, high nibbles 16..31
#pragma unroll
        for (uint32_t i = 0; i < 2; ++i) {
            const uint32_t q = r.q[T == T_Q4_0 ? j : j % 4u][i];
            const uint32_t off = 0xe408u;  // - 1032
            w[2u * i] = pk_add16((q & 0x000f000fu) | 0x64006400u, h16x2(off));
            w[2u * i + 1u] = pk_add16(((q >> 8) & 0x000f000fu) | 0x64006400u, h16x2(off));
            w[4u + 2u * i] = pk_add16(((q >> 4) & 0x000f000fu) | 0x64006400u, h16x2(off));
            w[5u + 2u * i] = pk_add16(((q >> 12) & 0x000f000fu) | 0x64006400u, h16x2(off));
        }
        if constexpr (T == T_Q4_0) ds[0] = ds[1] = half_of(hd.d, j);
        else ds[0] = ds[1] = half_bits_to_float(r.dm[j % 4u] & 0xffffu);
    }
    b[0] = frag4(w[0], w[1], w[2], w[3]);
    b[1] = frag4(w[4], w[5], w[6], w[7]);
}

// Takes a superblock's header.  kSuper: the B fragment of its mins (16 m_j as
// fp16 codes), the factor that brings the accumulator from the units of the
// superblock before (dcur) to this one's, and the mins' coefficient there.  A
// zero d keeps the units and zeroes the scales.
template <int T, bool UNITS>
__device__ __forceinline__ void whead(const WRaw<T>& r, WHead<T>& hd, uint32_t kq, f16x8& mins,
                                      float& dcur, float& rescale, float& cmin) {
    using W = WTraits<T, UNITS>;
    if constexpr (T == T_Q4_K || T == T_Q5_K) {
        const float d = half_bits_to_float(r.h[0] & 0xffffu);
        const float dmin = half_bits_to_float(r.h[0] >> 16);
        const bool zero = W::kUnits && d == 0.0f;
        const uint32_t keep = zero ? 0u : 0xffffffffu;
        // 6-bit scales and mins of groups 0..3 and 4..7 (src/quantized_linear.cpp:176-188)
        hd.sc[0] = r.h[1] & 0x3f3f3f3fu & keep;
        hd.sc[1] = ((r.h[3] & 0x0f0f0f0fu) | ((r.h[1] >> 2) & 0x30303030u)) & keep;
        const uint32_t m0 = r.h[2] & 0x3f3f3f3fu;
        const uint32_t m1 = ((r.h[3] >> 4) & 0x0f0f0f0fu) | ((r.h[2] >> 2) & 0x30303030u);
        if constexpr (W::kUnits) {
            mins = frag4(__builtin_amdgcn_perm(0u, m0, 0x0c010c00u) << 4,
                         __builtin_amdgcn_perm(0u, m0, 0x0c030c02u) << 4,
                         __builtin_amdgcn_perm(0u, m1, 0x0c010c00u) << 4,
                         __builtin_amdgcn_perm(0u, m1, 0x0c030c02u) << 4);
            const float dn = zero ? dcur : d, inv = 1.0f / dn;
            rescale = __fmul_rn(dcur, inv);
            cmin = __fmul_rn(__fmul_rn(-2.0f, dmin), inv);  // 2^5 (sums) / 2^4 (16 m_j)
            dcur = dn;
        } else {
            hd.d = d * 0x1p12f;
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {  // 16 d sc_j - dmin m_j of group j = 2 i + kq
                if constexpr (T == T_Q5_K) hd.qh[i] = r.qh[i];
                const uint32_t sh = 16u * (i & 1u) + 8u * kq;
                const float m = static_cast<float>(((i < 2u ? m0 : m1) >> sh) & 0xffu);
                const float sc = static_cast<float>((hd.sc[i / 2u] >> sh) & 0xffu);
                hd.cn[i] = __fmaf_rn(-dmin, m, __fmul_rn((T == T_Q5_K ? 16.0f : 8.0f) * d, sc));
            }
        }
    } else if constexpr (T == T_Q6_K) {
#pragma unroll
        for (int i = 0; i < 4; ++i) hd.sc[i] = r.sc[i];
        hd.d = half_bits_to_float(r.d);
    } else if constexpr (T == T_Q8_0 || T == T_Q4_0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) hd.d[i] = r.d[i];
    }
}

// ---------------------------------------------------------------------------
// Tiles.

struct TileRef {
    uint32_t e, base, rows;  // expert, first grouped row, valid rows (at most 64)
};

__device__ __forceinline__ bool tile_ref(const MoePrefillArgs& a, uint32_t tile, TileRef& r) {
    if (tile >= a.n_tiles[0]) return false;
    const uint32_t code = __builtin_amdgcn_readfirstlane(a.tiles[tile]);
    r.e = code >> 16;
    const uint32_t lo = __builtin_amdgcn_readfirstlane(a.offsets[r.e]);
    const uint32_t hi = __builtin_amdgcn_readfirstlane(a.offsets[r.e + 1]);
    r.base = lo + (code & 0x7fffu) * 32u;
    const uint32_t most = code & kTileBig ? kGemmTileM : 32u;
    r.rows = hi - r.base < most ? hi - r.base : most;
    return true;
}

// Workgroups go to the 8 XCDs round robin by linear id.  Block L runs on XCD
// L % 8; on each XCD, the blocks walk its tiles (tile % 8 == XCD) with all
// `nb` row blocks of one tile next to each other, so a tile's activations
// are fetched into that XCD's L2 once.  The tiles of one expert have consecutive
// numbers and so lie on different XCDs, each of which fetches the expert's weights
// again: 512 tokens of skewed load read 1.46 (gate/up) and 2.11 (down) times the
// bytes that one fetch of everything would take.
__device__ __forceinline__ void xcd_tile(uint32_t nb, uint32_t& tile, uint32_t& yb) {
    const uint32_t L = blockIdx.x, xcd = L % 8u, slot = L / 8u;
    tile = 8u * (slot / nb) + xcd;
    yb = slot % nb;
}

constexpr uint32_t kRowsN = 128;    // output rows per matrix and workgroup (4 waves x 32)
constexpr uint32_t kStageRow = 128; // bytes of one stage of one row: 32 values, hi then lo

struct GemmShared {
    uint8_t st[2][kGemmTileM * kStageRow];  // two stages of activations
    uint8_t xs[2][kGemmTileM * 32u];        // group sums of two superblocks: 8 hi, 8 lo
    uint32_t arow[kGemmTileM], oslot[kGemmTileM];
    float scale[kGemmTileM];
    uint32_t far;  // down: some row's chunk scales are far apart
};

// Maximum of |v| over each 32-lane half, in all its lanes (as unsigned bits, whose
// zero identity lets each DPP step fold into the maximum; NaN sorts last and
// gives the scale of an infinity).
__device__ __forceinline__ float half_wave_max(float v) {
    uint32_t u = __float_as_uint(v) & 0x7fffffffu;
    u = max(u, dpp_u0max<0xb1>(u));
    u = max(u, dpp_u0max<0x4e>(u));
    u = max(u, dpp_u0max<0x141>(u));
    u = max(u, dpp_u0max<0x140>(u));
    const auto s = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return __uint_as_float(max(s[0], s[1]));
}

// MT x 32 assignments of a tile.  DUAL: gate and up rows n0 .. n0 + 127 over x, SwiGLU,
// activations split for the down GEMM; otherwise down rows n0 .. n0 + 255 over the
// activations, each output row to its (token, route) slot.  FAR: some chunk's scale
// lies more than 2^24 below its row's, and the halves come down in two steps (which in
// every tile would cost 0.5 to 2%).
template <int T, bool UNITS, bool DUAL, int MT, bool FAR = false>
__device__ __forceinline__ void gemm_tile(const MoePrefillArgs& a, const TileRef& tr, uint32_t n0,
                                          GemmShared& sh) {
    using W = WTraits<T, UNITS>;
    const MoeDecodeArgs& L = a.layer;
    const uint32_t kdim = DUAL ? L.hidden : L.ffn, ndim = DUAL ? L.ffn : L.hidden;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t ln = lane % 32u, kq = lane / 32u;
    const uint32_t nst = kdim / 32u;
    // superblocks sb0 .. nsb - 1 of K: all, or this workgroup's share (dense GEMMs)
    const uint32_t all = kdim / 256u, parts_k = DUAL ? 1u : a.k_parts;
    const uint32_t sb0 = blockIdx.y * all / parts_k, nsb = (blockIdx.y + 1u) * all / parts_k;

    // weights
    const bool shared = tr.e >= L.n_experts;  // the shared expert (variant 1): its own tensors
    const uint32_t rnb = kdim / Fmt<T>::BE;
    WSrc<T> ws[2];
    if constexpr (DUAL) {
        const uint64_t nblk = static_cast<uint64_t>(L.ffn) * rnb, b0 = static_cast<uint64_t>(n0) * rnb;
        ws[0] = wsrc<T>(shared ? L.shared_gate : L.gate + static_cast<uint64_t>(tr.e) * L.gate_slice, nblk, b0);
        ws[1] = wsrc<T>(shared ? L.shared_up : L.up + static_cast<uint64_t>(tr.e) * L.up_slice, nblk, b0);
    } else {
        const uint8_t* base = shared ? L.shared_down : L.down + static_cast<uint64_t>(tr.e) * L.down_slice;
        const uint64_t nblk = static_cast<uint64_t>(L.hidden) * rnb;
        ws[0] = wsrc<T>(base, nblk, static_cast<uint64_t>(n0) * rnb);
        ws[1] = wsrc<T>(base, nblk, static_cast<uint64_t>(n0 + kRowsN) * rnb);
    }
    const uint32_t blk = (wave * 32u + ln) * rnb;  // this lane's row's first block
    WRaw<T> raw[2];
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
        wload_head<T>(ws[i], blk, sb0, kq, raw[i]);
#pragma unroll
        for (uint32_t j = 0; j < (T == T_Q8_0 || T == T_Q4_1 ? 4u : 8u); ++j) wload_step<T>(ws[i], blk, sb0, j, kq, raw[i]);
    }

    // activations: thread t moves piece t % 8 (16 bytes) of rows t / 8 (+ 32)
    const uint16_t* parts = DUAL ? a.x_parts : a.act_parts;
    const float* sums = DUAL ? a.x_sums : a.act_sums;
    const uint32_t pr = tid / 8u, pc = tid % 8u;
    const uint16_t* asrc[MT];
    const float* csrc[MT];   // down: the chunk scales of the piece's row
    float cinv[MT];
    uint32_t adst[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const uint32_t row = pr + 32u * i;
        asrc[i] = parts + static_cast<uint64_t>(sh.arow[row]) * kdim * 2u + pc * 8u;
        adst[i] = row * kStageRow + ((pc ^ (row & 7u)) * 16u);
        csrc[i] = DUAL ? nullptr : a.act_scale + static_cast<uint64_t>(sh.arow[row]) * nst;
        cinv[i] = DUAL ? 0.0f : 1.0f / sh.scale[row];
    }
    // register sets of stages in flight: with one row block there is room for eight,
    // which small batches need, where little else hides the loads' latency (77
    // tokens, 64 experts: gate/up 45 -> 42 us; 512 tokens 119 -> 117); Q5_K's down has
    // room for four
    constexpr uint32_t NS = MT == 2 || FAR ? 2u : T == T_Q5_K && !DUAL ? 4u : 8u;
    u32x4_t av[NS][MT];
    float ac[NS][MT];
    const uint32_t last = 8u * nsb - 1u;
    auto load_act = [&](uint32_t set, uint32_t s) {  // past the end: the last stage again
        const uint32_t st = s < last ? s : last;
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            av[set][i] = *reinterpret_cast<const u32x4_t*>(asrc[i] + st * 64u);
            if constexpr (!DUAL) ac[set][i] = csrc[i][st];
        }
    };
    auto store_act = [&](uint32_t set, uint32_t buf) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            u32x4_t v = av[set][i];
            if constexpr (!DUAL) {  // from the chunk's scale to the row's (a power of two, at most 1)
                const float r = ac[set][i] * cinv[i];
                if constexpr (FAR) {  // FP16 ends at 2^-24: the rest as a second factor
                    const bool far = r < 0x1p-24f;
                    const f16x2 g = __builtin_bit_cast(f16x2, far ? 0x00010001u : 0x3c003c00u);  // 2^-24, 1
                    const _Float16 f = static_cast<_Float16>(far ? r * 0x1p24f : r);
                    const f16x2 ff = {f, f};
#pragma unroll
                    for (int k = 0; k < 4; ++k) v[k] = pk_mul_f16(pk_mul_f16(v[k], ff), g);
                } else {
                    const _Float16 f = static_cast<_Float16>(r);
                    const f16x2 ff = {f, f};
#pragma unroll
                    for (int k = 0; k < 4; ++k) v[k] = pk_mul_f16(v[k], ff);
                }
            }
            *reinterpret_cast<u32x4_t*>(sh.st[buf] + adst[i]) = v;
        }
    };
    // group sums: thread t takes groups 2 (t % 4), + 1 of row t / 4; with one row block
    // the upper half of the threads has none.  It stores row 0's sums to the rows that
    // nobody reads all the same: a branch here would split the unrolled superblock, and
    // the values held across it do not fit the registers (Q4_1: 61 spilled with one row
    // block, 340 with two; none without the branch).  kUnits, with no FMA per step,
    // fits better with it (208 registers against 256 and 25 spilled).
    const uint32_t dr = tid / 4u, sr = dr < 32u * MT ? dr : 0u, sg = 2u * (tid % 4u);
    const float* ssrc = W::kMins ? sums + static_cast<uint64_t>(sh.arow[sr]) * nst + sg : nullptr;
    const float sinv = W::kMins ? (W::kMinsF32 ? 1.0f : 0x1p-5f) / sh.scale[sr] : 0.0f;
    float2 sv = make_float2(0.0f, 0.0f);
    auto load_sums = [&](uint32_t sb) {
        if constexpr (W::kMins) sv = *reinterpret_cast<const float2*>(ssrc + 8u * (sb < nsb ? sb : nsb - 1u));
    };
    auto store_sums = [&](uint32_t buf) {
        if (W::kUnits && tid >= 128u * MT) return;
        if constexpr (W::kMinsF32) {
            *reinterpret_cast<float2*>(sh.xs[buf] + dr * 32u + sg * 4u) = make_float2(sv.x * sinv, sv.y * sinv);
        } else if constexpr (W::kMins) {
            uint32_t hi, lo;
            split_pair(sv.x * sinv, sv.y * sinv, hi, lo);
            *reinterpret_cast<uint32_t*>(sh.xs[buf] + dr * 32u + sg * 2u) = hi;
            *reinterpret_cast<uint32_t*>(sh.xs[buf] + dr * 32u + 16u + sg * 2u) = lo;
        }
    };
    // A fragments: piece (plane, 2 kq + h or 2 h + kq) of row ln (+ 32)
    const uint32_t fx = ((W::kHalfRuns ? 2u * kq : kq) ^ (ln & 7u)) * 16u;
    auto afrag = [&](uint32_t buf, uint32_t m, uint32_t plane, uint32_t h) {
        const uint32_t p = (4u * plane + (W::kHalfRuns ? h : 2u * h)) * 16u;
        return __builtin_bit_cast(f16x8, *reinterpret_cast<const u32x4_t*>(
                                             sh.st[buf] + (ln + 32u * m) * kStageRow + (fx ^ p)));
    };
    auto sfrag = [&](uint32_t buf, uint32_t m) {
        return __builtin_bit_cast(f16x8, *reinterpret_cast<const u32x4_t*>(
                                             sh.xs[buf] + (ln + 32u * m) * 32u + kq * 16u));
    };

    load_act(0u, 8u * sb0);
    load_sums(sb0);
#pragma unroll
    for (uint32_t i = 1; i < NS; ++i) load_act(i, 8u * sb0 + i);
    store_act(0u, 0u);
    store_sums(sb0 & 1u);
    load_act(0u, 8u * sb0 + NS);
    __syncthreads();

    // sums over a superblock: Q5_K the high and the low halves' apart, Q4_K one
    constexpr uint32_t kSums = MT == 1 && W::kSuper && !W::kUnits ? (T == T_Q5_K ? 2u : 1u) : 0u;
    f32x16 acc[MT][2], sum[2][2];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m][0] = acc[m][1] = f32x16{};
    float dcur[2] = {1.0f, 1.0f};
    WHead<T> hd[2];
    for (uint32_t sb = sb0; sb < nsb; ++sb) {
        const uint32_t bn = sb + 1u < nsb ? sb + 1u : nsb - 1u, sbuf = sb & 1u;
        {
            f16x8 mins[2];
            float rescale[2], cmin[2];
#pragma unroll
            for (uint32_t i = 0; i < 2; ++i) {
                whead<T, UNITS>(raw[i], hd[i], kq, mins[i], dcur[i], rescale[i], cmin[i]);
                wload_head<T>(ws[i], blk, bn, kq, raw[i]);
            }
            if constexpr (W::kUnits) {
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    const f16x8 s = sfrag(sbuf, m);
#pragma unroll
                    for (uint32_t i = 0; i < 2; ++i) {
                        const f32x16 p = mfma(s, mins[i], f32x16{});
#pragma unroll
                        for (uint32_t r = 0; r < 16; ++r)
                            acc[m][i][r] = __builtin_fmaf(p[r], cmin[i], __fmul_rn(acc[m][i][r], rescale[i]));
                    }
                }
            }
            load_sums(sb + 1u);
        }
#pragma unroll
        for (uint32_t j = 0; j < 8u; ++j) {
            const uint32_t s = 8u * sb + j, buf = j & 1u;
            f16x8 b[2][2];
            float ds[2][2];
#pragma unroll
            for (uint32_t i = 0; i < 2; ++i) wfrag<T, UNITS>(raw[i], hd[i], j, b[i], ds[i]);
            if constexpr (T == T_Q4_1) {  // the mins of groups 2 i + kq
#pragma unroll
                for (uint32_t i = 0; i < 2; ++i) {
                    const float m = __fmaf_rn(8.0f, ds[i][0], half_bits_to_float(raw[i].dm[j % 4u] >> 16));
                    hd[i].cn[j / 2u] = j & 1u ? (kq ? m : hd[i].cn[j / 2u]) : m;
                }
            }
            if constexpr (W::kUnits) {
#pragma unroll
                for (uint32_t h = 0; h < 2; ++h)
#pragma unroll
                    for (int m = 0; m < MT; ++m) {
                        const f16x8 lo = afrag(buf, m, 1u, h), hi = afrag(buf, m, 0u, h);
                        acc[m][0] = mfma(lo, b[0][h], acc[m][0]);
                        acc[m][1] = mfma(lo, b[1][h], acc[m][1]);
                        acc[m][0] = mfma(hi, b[0][h], acc[m][0]);
                        acc[m][1] = mfma(hi, b[1][h], acc[m][1]);
                    }
            } else if constexpr (kSums) {
                // low and high of one fragment, then of the other; with two sums, in the
                // superblock's last step both low ones first, so that their sums go into the
                // accumulator while the high products end
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) {
                    const bool lows = kSums == 2u && j == 7u;
                    const uint32_t h = lows ? k & 1u : k / 2u, p = lows ? k < 2u : !(k & 1u), q = p & (kSums - 1u);
                    const f16x8 f = afrag(buf, 0u, p, h);
#pragma unroll
                    for (uint32_t i = 0; i < 2; ++i)
                        sum[i][q] = mfma(f, b[i][h], j == 0u && k < kSums ? f32x16{} : sum[i][q]);
                }
                if (j == 7u) {
#pragma unroll
                    for (uint32_t q = 0; q < kSums; ++q)
#pragma unroll
                        for (uint32_t i = 0; i < 2; ++i)
#pragma unroll
                            for (uint32_t r = 0; r < 16; ++r)
                                acc[0][i][r] = __builtin_fmaf(hd[i].d, sum[i][kSums - 1u - q][r], acc[0][i][r]);
                }
            } else {
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    f32x16 P[2];
#pragma unroll
                    for (uint32_t k = 0; k < 4; ++k) {
                        // group 32: both low halves, then both high ones, so that few roundings are
                        // at full size; group 16: low and high of one fragment at a time
                        const bool g32 = W::kGroup == 32u;
                        const uint32_t h = g32 ? k & 1u : k / 2u, p = g32 ? k < 2u : !(k & 1u);
                        const f16x8 f = afrag(buf, m, p, h);
#pragma unroll
                        for (uint32_t i = 0; i < 2; ++i)
                            P[i] = mfma(f, b[i][h], (g32 ? k : k & 1u) == 0u ? f32x16{} : P[i]);
                        if (k == 3u || (!g32 && k == 1u)) {
#pragma unroll
                            for (uint32_t i = 0; i < 2; ++i)
#pragma unroll
                                for (uint32_t r = 0; r < 16; ++r)
                                    acc[m][i][r] = __builtin_fmaf(ds[i][h], P[i][r], acc[m][i][r]);
                        }
                    }
                }
            }
            if constexpr (W::kMinsF32) {
                if (j == 7u) {
#pragma unroll
                    for (int m = 0; m < MT; ++m)
#pragma unroll
                        for (uint32_t g = 0; g < 4; ++g) {  // groups 2 g + kq
                            const float av = *reinterpret_cast<const float*>(
                                sh.xs[sbuf] + (ln + 32u * m) * 32u + (2u * g + kq) * 4u);
                            acc[m][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(av, hd[0].cn[g], acc[m][0], 0, 0, 0);
                            acc[m][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(av, hd[1].cn[g], acc[m][1], 0, 0, 0);
                        }
                }
            }
#pragma unroll
            for (uint32_t i = 0; i < 2; ++i) wreload<T>(ws[i], blk, sb, bn, j, kq, raw[i]);
            store_act((j + 1u) % NS, buf ^ 1u);
            load_act((j + 1u) % NS, s + 1u + NS);
            if (j == 4u) store_sums(sbuf ^ 1u);
            __syncthreads();
            // Q4_K: keeps the next step's decoding behind this one's products (8 registers
            // spill without; Q5_K does not spill and is 4% slower with it)
            if constexpr (kSums == 1u) __builtin_amdgcn_sched_barrier(0);
        }
    }

    // results: the accumulators' units are d 2^24 s (kSuper) or s (the row's scale)
    const float u0 = W::kUnits ? dcur[0] * 0x1p24f : 1.0f, u1 = W::kUnits ? dcur[1] * 0x1p24f : 1.0f;
    if constexpr (DUAL) {
        // SwiGLU g / (1 + exp(-g)) * u (src/qwen3_moe_runner.cpp:682-684, and variant 1's
        // silu(g) * u, src/qwen35_runner.cpp:111-123) with the hardware exp2 and
        // reciprocal, as the decode path; the values split as the down GEMM's
        // operands: the wave's 32 columns of a row are one chunk.  (With the libm
        // expf, IEEE division and 64-bit addresses this part took nearly half of
        // the kernel's vector instructions: 526 -> 494 us at 4096 tokens.)
        const uint32_t col = n0 + wave * 32u + ln, chunk = col / 32u, nch = ndim / 32u;
        const uint32_t at = (ln & 24u) | kPairOrder(ln & 7u);
        const bool dmins = L.down_type == T_Q4_K || L.down_type == T_Q5_K || L.down_type == T_Q4_1;
        // this lane's place in row 0 of the tile's rows; rows are nch stages apart
        const uint64_t rc0 = static_cast<uint64_t>(tr.base) * nch + chunk;
        uint16_t* pd = a.act_parts + rc0 * 64u + at;
        float* cd = a.act_scale + rc0;
        float* sd = a.act_sums + rc0;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
#pragma unroll
            for (uint32_t r = 0; r < 16; ++r) {
                const uint32_t row = 32u * m + (r / 4u) * 8u + kq * 4u + (r % 4u);
                const float s = sh.scale[row];
                const float g = acc[m][0][r] * (u0 * s), u = acc[m][1][r] * (u1 * s);
                const float v = (g * __builtin_amdgcn_rcpf(1.0f + __expf(-g))) * u;
                float cs, cinv2;
                split_scale(half_wave_max(v), cs, cinv2);
                const float w = v * cinv2;
                const _Float16 h = static_cast<_Float16>(w);
                const _Float16 l = static_cast<_Float16>(w - static_cast<float>(h));
                float gs = 0.0f;
                if (dmins) gs = static_cast<float>(group_sum<32>(static_cast<double>(v)));  // uniform
                if (row < tr.rows) {
                    const uint32_t off = row * nch;
                    pd[off * 64u] = __builtin_bit_cast(uint16_t, h);
                    pd[off * 64u + 32u] = __builtin_bit_cast(uint16_t, l);
                    if (ln == 31u) {
                        cd[off] = cs;
                        if (dmins) sd[off] = gs;
                    }
                }
            }
        }
    } else {
        float* out = a.out + blockIdx.y * a.out_part;
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (uint32_t r = 0; r < 16; ++r) {
                const uint32_t row = 32u * m + (r / 4u) * 8u + kq * 4u + (r % 4u);
                if (row < tr.rows) {
                    const float s = sh.scale[row];
                    float* o = out + static_cast<uint64_t>(sh.oslot[row]) * ndim + n0 + wave * 32u + ln;
                    o[0] = acc[m][0][r] * u0 * s;
                    o[kRowsN] = acc[m][1][r] * u1 * s;
                }
            }
    }
}

template <int T, bool UNITS, bool DUAL>
__global__ __launch_bounds__(256, 2) void k_expert_gemm(MoePrefillArgs a) {
    __shared__ __attribute__((aligned(16))) GemmShared sh;
    const MoeDecodeArgs& L = a.layer;
    const uint32_t ndim = DUAL ? L.ffn : L.hidden;
    const uint32_t nblk = DUAL ? kRowsN : 2u * kRowsN;  // output rows per workgroup
    uint32_t tile, yb;
    xcd_tile(ndim / nblk, tile, yb);
    TileRef tr;
    if (!tile_ref(a, tile, tr)) return;  // uniform
    const uint32_t tid = threadIdx.x;
    if (tid < kGemmTileM) {
        const uint32_t i = tid < tr.rows ? tid : tr.rows - 1u;  // absent rows repeat a real one
        const uint32_t slot = a.perm[tr.base + i];  // token * top_k + route
        const uint32_t row = DUAL ? slot / (L.top_k + L.variant) : tr.base + i;
        sh.arow[tid] = row;
        sh.oslot[tid] = slot;
        if constexpr (DUAL) sh.scale[tid] = a.x_scale[row];
    }
    if constexpr (!DUAL) {  // a row's scale: the largest of its chunks'
        if (tid == 0u) sh.far = 0u;
        __syncthreads();
        const uint32_t row = tid / 4u, nch = L.ffn / 32u;
        const float* cs = a.act_scale + static_cast<uint64_t>(sh.arow[row]) * nch;
        // the least scale of a chunk that is not zero, as bits past kZeroScale's (a zero
        // chunk's wrap around)
        const uint32_t past = __float_as_uint(kZeroScale) + 1u;
        float m = 0.0f;
        uint32_t least = ~0u;
        for (uint32_t c = tid % 4u; c < nch; c += 4u) {
            const float s = cs[c];
            m = fmaxf(m, s);
            least = min(least, __float_as_uint(s) - past);
        }
        m = fmaxf(m, dpp<0xb1>(m));
        m = fmaxf(m, dpp<0x4e>(m));
        // (below 2^-84 what has the zero scale may not be nothing to the row; at 2^-102 and
        // below no scale lies 2^24 under it)
        if (m > 0x1p-102f && (m < 0x1p-84f || least < __float_as_uint(m * 0x1p-24f) - past)) sh.far = 1u;
        if (tid % 4u == 0u) sh.scale[row] = m;
    }
    __syncthreads();
    if constexpr (!DUAL) {
        if (__builtin_amdgcn_readfirstlane(sh.far)) {  // outliers in the activations
            if (tr.rows > 32u) gemm_tile<T, UNITS, false, 2, true>(a, tr, yb * nblk, sh);
            else gemm_tile<T, UNITS, false, 1, true>(a, tr, yb * nblk, sh);
            return;
        }
    }
    if (tr.rows > 32u) {
        gemm_tile<T, UNITS, DUAL, 2>(a, tr, yb * nblk, sh);
    } else {
        gemm_tile<T, UNITS, DUAL, 1>(a, tr, yb * nblk, sh);
    }
}

template <int T, bool DUAL>
hipError_t expert_gemm_t(const MoePrefillArgs& a, hipStream_t s) {
    const MoeDecodeArgs& L = a.layer;
    const uint32_t nb = DUAL ? L.ffn / kRowsN : L.hidden / (2u * kRowsN);
    const uint32_t blocks = 8u * ((a.max_tiles + 7u) / 8u) * nb;  // xcd_tile's layout
    const dim3 grid(blocks, DUAL ? 1u : a.k_parts);
    if constexpr (T == T_Q4_K && !DUAL) {
        if (a.precise) {
            hipLaunchKernelGGL((k_expert_gemm<T, false, DUAL>), grid, dim3(256), 0, s, a);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((k_expert_gemm<T, T == T_Q4_K, DUAL>), grid, dim3(256), 0, s, a);
    return hipGetLastError();
}

template <bool DUAL>
hipError_t expert_gemm(uint32_t type, const MoePrefillArgs& a, hipStream_t s) {
    switch (type) {
        case T_Q4_K: return expert_gemm_t<T_Q4_K, DUAL>(a, s);
        case T_Q5_K: return expert_gemm_t<T_Q5_K, DUAL>(a, s);
        case T_Q6_K: return expert_gemm_t<T_Q6_K, DUAL>(a, s);
        case T_Q8_0: return expert_gemm_t<T_Q8_0, DUAL>(a, s);
        case T_Q4_0: return expert_gemm_t<T_Q4_0, DUAL>(a, s);
        case T_Q4_1: return expert_gemm_t<T_Q4_1, DUAL>(a, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

uint32_t moe_prefill_tile_wgs(uint32_t hidden, uint32_t ffn) {
    return ffn / kRowsN > hidden / (2u * kRowsN) ? ffn / kRowsN : hidden / (2u * kRowsN);
}

hipError_t launch_expert_gate_up(const MoePrefillArgs& a, hipStream_t s) {
    return expert_gemm<true>(a.layer.gate_type, a, s);
}

hipError_t launch_expert_down(const MoePrefillArgs& a, hipStream_t s) {
    return expert_gemm<false>(a.layer.down_type, a, s);
}

}  // namespace pk
