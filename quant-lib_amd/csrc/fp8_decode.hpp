// fp8_decode.hpp -- FP8 codes to fp32 and binary16 (the reference's decoding and the
// OCP one), shared by the codec and the FP8-weight GEMMs.
#pragma once

#include "ql_common.hpp"
#include "quantlib_amd.h"

namespace ql {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

template <int FMT>
__device__ __forceinline__ float dec_ref(uint32_t q) {
    constexpr int MB = FMT == QL_FP8_E4M3 ? 3 : 2, BIAS = FMT == QL_FP8_E4M3 ? 7 : 15;
    const uint32_t e = (q >> MB) & (FMT == QL_FP8_E4M3 ? 0xFu : 0x1Fu);
    const uint32_t m = q & ((1u << MB) - 1u);
    const uint32_t bits = ((q & 0x80u) << 24) | ((e + 127u - BIAS) << 23) | (m << (23 - MB));
    return (e == 0 && m == 0) ? 0.0f : __uint_as_float(bits);
}

// the two bytes of w's low (HI = false) or high 16-bit word
template <int FMT, bool HI = false>
__device__ __forceinline__ float2v dec_ocp2(uint32_t w) {
    if constexpr (FMT == QL_FP8_E4M3)
        return __builtin_amdgcn_cvt_pk_f32_fp8((int)w, HI);
    else
        return __builtin_amdgcn_cvt_pk_f32_bf8((int)w, HI);
}

// two codes (the low or high half of w) -> two binary16, exact (every E4M3 / E5M2
// value is a binary16 value; the scale operand 1.0 leaves them as decoded)
template <int FMT, bool HI = false>
__device__ __forceinline__ half2v dec_ocp2_h(uint32_t w) {
    if constexpr (FMT == QL_FP8_E4M3)
        return __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, HI);
    else
        return __builtin_amdgcn_cvt_scalef32_pk_f16_bf8(w, 1.0f, HI);
}

// bytes of 4 reference-mode codes whose reference decode differs from the OCP
// decode (bit 7 of each byte of the result): E4M3 exponent 0 with a non-zero
// mantissa (the reference reads it as a normal number) and |code| 0x7F (the
// reference's 480, OCP's NaN); E5M2 exponent 0 with a non-zero mantissa and
// exponent 31 (finite in the reference).  With l = |code| (7 bits) per byte,
// l + 0x7F has bit 7 iff l >= 1, 0x87 - l (or 0x83 - l) iff l <= 7 (l <= 3), and
// l + 0x01 (l + 0x04) iff l == 0x7F (l >= 0x7C); none of these carries or borrows
// across bytes.  The caller masks the OR of several words with 0x80808080.
template <int FMT>
__device__ __forceinline__ uint32_t ref_special(uint32_t w) {
    const uint32_t l = w & 0x7F7F7F7Fu;
    const uint32_t ge1 = l + 0x7F7F7F7Fu;
    const uint32_t le_m = (FMT == QL_FP8_E4M3 ? 0x87878787u : 0x83838383u) - l;
    const uint32_t top = l + (FMT == QL_FP8_E4M3 ? 0x01010101u : 0x04040404u);
    return (ge1 & le_m) | top;
}

// 16 codes -> two fp16 fragments of binary16(decode(code) * inv).  The hardware
// decode is exact for every OCP code; in reference mode it is used when none of a
// lane's 16 codes is one of the codes whose reference value differs (the reference
// encoder only writes such a code for a NaN input) and the lane falls back to the
// bitwise reference decode otherwise.  SCALED = false leaves the scale out (the
// caller applies it to the accumulated products): every FP8 value is exact in
// binary16, so the fragments then hold the decoded codes themselves, converted
// two at a time straight to binary16 (callers keep reference-mode E5M2, whose
// exponent-31 codes exceed the binary16 range, on SCALED = true).
template <int FMT, int MODE, bool SCALED>
__device__ __forceinline__ void dequant16(uint4 codes, float inv, half8& lo, half8& hi) {
    const uint32_t w[4] = {codes.x, codes.y, codes.z, codes.w};
    if constexpr (!SCALED) {
        // straight to binary16: one conversion per two codes
        half2v h[8];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            h[2 * j] = dec_ocp2_h<FMT>(w[j]);
            h[2 * j + 1] = dec_ocp2_h<FMT, true>(w[j]);
        }
        if constexpr (MODE == QL_FP8_MODE_REFERENCE) {
            const uint32_t special = (ref_special<FMT>(w[0]) | ref_special<FMT>(w[1]) | ref_special<FMT>(w[2]) |
                                      ref_special<FMT>(w[3])) & 0x80808080u;
            if (special) {
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    h[e >> 1][e & 1] = (_Float16)dec_ref<FMT>((w[e >> 2] >> (8 * (e & 3))) & 0xFFu);
            }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            lo[e] = h[e >> 1][e & 1];
            hi[e] = h[4 + (e >> 1)][e & 1];
        }
        return;
    }
    float f[16];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float2v a = dec_ocp2<FMT>(w[j]);
        const float2v b = dec_ocp2<FMT, true>(w[j]);
        f[4 * j] = a[0];
        f[4 * j + 1] = a[1];
        f[4 * j + 2] = b[0];
        f[4 * j + 3] = b[1];
    }
    if constexpr (MODE == QL_FP8_MODE_REFERENCE) {
        const uint32_t special = (ref_special<FMT>(w[0]) | ref_special<FMT>(w[1]) | ref_special<FMT>(w[2]) |
                                  ref_special<FMT>(w[3])) & 0x80808080u;
        if (special) {
#pragma unroll
            for (int e = 0; e < 16; ++e) f[e] = dec_ref<FMT>((w[e >> 2] >> (8 * (e & 3))) & 0xFFu);
        }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        lo[e] = (_Float16)(f[e] * inv);
        hi[e] = (_Float16)(f[8 + e] * inv);
    }
}

}  // namespace ql
