// Block scales, codes and decoding of NVFP4, shared by its kernels.
#pragma once
#include "common.h"

namespace mo {

// E4M3 byte of a block scale bs = bmax / gs6 (0 -> 1.0).  When the quotient is NaN because of
// an invalid operation (0/0, inf/inf) the x86 reference produces the negative default NaN and
// therefore the byte 0xFF; a NaN that comes from a NaN operand keeps that operand's (positive)
// sign and gives 0x7F.  `cap` is +inf for the reference's cast (a quotient above E4M3's range
// becomes the NaN byte) or 448 to saturate instead (flag MO_FLAG_SATURATE_BLOCK_SCALE).
__device__ __forceinline__ uint32_t block_scale_byte(float bmax, float gs6,
                                                     float cap = __builtin_inff()) {
    float bs = bmax / gs6;
    if (bs == 0.0f) bs = 1.0f;
    if (bs != bs) return (bmax != bmax || gs6 != gs6) ? 0x7Fu : 0xFFu;
    return f32_to_e4m3<false>(bs < cap ? bs : cap);
}

// bits of the `opts` kernel argument
constexpr int kOptForceExact = 1, kOptSaturateScale = 2;
__device__ __forceinline__ float scale_cap(int opts) {
    return (opts & kOptSaturateScale) ? 448.0f : __builtin_inff();
}

typedef float f32x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ void decode8(uint32_t codes, float s, float (&v)[8]) {
#define MO_DEC(SEL)                                                                     \
    {                                                                                   \
        f32x2_t p = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(codes, 1.0f, SEL);         \
        v[2 * SEL] = (p.x + 0.0f) * s;                                                  \
        v[2 * SEL + 1] = (p.y + 0.0f) * s;                                              \
    }
    MO_DEC(0) MO_DEC(1) MO_DEC(2) MO_DEC(3)
#undef MO_DEC
}

// x / s for an element of type DT under a scale whose reciprocal r is correctly rounded
template <int DT>
__device__ __forceinline__ float quotient_of(float x, float s, float r) {
    if constexpr (DT == MO_F32) return exact_quotient(x, s, r);
    else return exact_quotient_short(x, s, r);
}

// Whether the reciprocal form of the quotient is exact for a block: scale in [2^-64, 2^10], abs-max
// finite, no quotient that overflows.
__device__ __forceinline__ bool nvfp4_scale_fast(float s, uint32_t bmax_bits, float r) {
    const uint32_t sb = f2u(s);
    return sb >= 0x1F800000u && sb <= 0x44800000u && bmax_bits < 0x7F800000u && u2f(bmax_bits) * r < 1.0e38f;
}

// The value one code unit of a block stands for in the quantize-dequantize: MODE 0 the threshold-ladder
// formula (block scale clamped at 448, values below 1e-5 replaced by 1), MODE 1 the packed format's.
template <int MODE>
__device__ __forceinline__ float nvfp4_unit(float bmax, float gs, float gs_safe) {
    if constexpr (MODE == 0) {
        float sc = bmax / (6.0f * gs_safe);
        if (sc == sc) sc = sc < 448.0f ? sc : 448.0f;
        const float s = round_e4m3<false>(sc) * gs;
        return s >= 1e-5f ? s : 1.0f;
    } else {
        return e4m3_to_f32(block_scale_byte(bmax, 6.0f * gs)) * gs;
    }
}

// Eight elements of a block with abs-max `bmax_bits` and unit `s`, quantised and dequantised.
template <int DT, int MODE>
__device__ __forceinline__ void nvfp4_qdq_chunk(const float (&v)[8], uint32_t bmax_bits, float s, float (&o)[8]) {
    const float r = 1.0f / s;
    if (nvfp4_scale_fast(s, bmax_bits, r)) {
        uint32_t c = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float a = v[2 * j], b = v[2 * j + 1];
            if constexpr (MODE == 0) { a = __builtin_fabsf(a); b = __builtin_fabsf(b); }
            c = fp4_pair(c, quotient_of<DT>(a, s, r), quotient_of<DT>(b, s, r), j);
        }
        decode8(c, s, o);
        if constexpr (MODE == 0) {
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = v[j] >= 0.0f ? o[j] : -o[j];
        }
        return;
    }
    keep_branch();
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        if constexpr (MODE == 0) {
            const float q = __builtin_fabsf(v[j]) / s;
            float lvl = 6.0f;
            lvl = q <= 5.0f ? 4.0f : lvl;
            lvl = q < 3.5f ? 3.0f : lvl;
            lvl = q <= 2.5f ? 2.0f : lvl;
            lvl = q < 1.75f ? 1.5f : lvl;
            lvl = q <= 1.25f ? 1.0f : lvl;
            lvl = q < 0.75f ? 0.5f : lvl;
            lvl = q <= 0.25f ? 0.0f : lvl;
            const float t = lvl * s;
            o[j] = v[j] >= 0.0f ? t : -t;
        } else {
            o[j] = e2m1_to_f32(f32_to_e2m1(v[j] / s)) * s;
        }
    }
}

// Codes of eight elements; `exact` forces the division.
template <int DT>
__device__ __forceinline__ uint32_t nvfp4_codes(const float (&v)[8], uint32_t bmax_bits, float s, bool exact) {
    const float r = 1.0f / s;
    uint32_t c = 0;
    if (!exact && nvfp4_scale_fast(s, bmax_bits, r)) {
        float q[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) q[j] = quotient_of<DT>(v[j], s, r);
        if constexpr (DT == MO_F32) {
            // The code keeps the sign of the quotient.  m smallest denormals over s round to a zero, which has
            // no sign here, where m <= s / 2; the short form may leave either neighbour.
            const float least = u2f((uint32_t)(0.5f * s));
#pragma unroll
            for (int j = 0; j < 8; ++j) q[j] = __builtin_fabsf(v[j]) > least ? q[j] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) c = fp4_pair(c, q[2 * j], q[2 * j + 1], j);
        return c;
    }
    keep_branch();
#pragma unroll
    for (int j = 0; j < 8; ++j) c |= f32_to_e2m1(v[j] / s) << (4 * j);
    return c;
}

__device__ __forceinline__ uint32_t chunk_absmax_bits(const float (&v)[8]) {
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        uint32_t t = f2u(v[j]) & 0x7FFFFFFFu;
        m = t > m ? t : m;
    }
    return m;
}

}  // namespace mo
