// Element rounding and block scales of the block floating point formats (MX and two-level), shared by the
// whole-tensor and the row-wise fake-quant kernels.
#pragma once
#include "common.h"

namespace mo {

// Nearest value of a small float format with M mantissa bits whose smallest normal number is
// 2^EMIN (below it the quantum stays 2^(EMIN - M)), saturating at fmax; `a` is non-negative,
// infinities and NaN give fmax.  Ties go to the even multiple of the quantum -- the value with
// the even index in the reference's tables -- or away from zero when TIES_AWAY.
template <int M, int EMIN, bool TIES_AWAY>
__device__ __forceinline__ float round_minifloat(float a, float fmax) {
    if constexpr (!TIES_AWAY) {
        // 2^(e + 23 - M), e the exponent of a or EMIN: its fp32 ulp is the quantum, so adding it
        // rounds a to a multiple of the quantum, ties to the even one, and subtracting it leaves that
        // multiple.  An infinite or NaN sum fails the comparison.
        uint32_t e = f2u(a) & 0x7F800000u;
        e = e > (uint32_t)(127 + EMIN) << 23 ? e : (uint32_t)(127 + EMIN) << 23;
        const float c = u2f(e + ((uint32_t)(23 - M) << 23));
        const float v = (a + c) - c;
        return a < fmax ? (v < fmax ? v : fmax) : fmax;
    }
    if (!(a < __builtin_inff())) return fmax;
    int e = (int)(f2u(a) >> 23) - 127;
    e = e > EMIN ? e : EMIN;
    const float t = __builtin_ldexpf(a, M - e);
    const float r = __builtin_floorf(t + 0.5f);
    const float v = __builtin_ldexpf(r, e - M);
    return v < fmax ? v : fmax;
}

// E5M2: round to nearest even with subnormals (quantum 2^-16), saturating at 57344; NaN stays.
__device__ __forceinline__ float round_e5m2_sat(float a) {
    if (a != a) return a;
    a = a < 57344.0f ? a : 57344.0f;
    int e = (int)(f2u(a) >> 23) - 127;
    e = e > -14 ? e : -14;
    const float v = __builtin_ldexpf(__builtin_rintf(__builtin_ldexpf(a, 2 - e)), e - 2);
    return v < 57344.0f ? v : 57344.0f;
}

template <int FMT>
__device__ __forceinline__ float convert_elem(float a) {  // a >= 0 (or NaN)
    if constexpr (FMT == MO_EF_E4M3) return round_e4m3<true>(a);
    else if constexpr (FMT == MO_EF_E5M2) return round_e5m2_sat(a);
    else if constexpr (FMT == MO_EF_INT8) {
        const float q = __builtin_rintf(a);
        return q > 127.0f ? 127.0f : q;  // NaN stays NaN
    }
    else if constexpr (FMT == MO_EF_E0M3) return round_minifloat<3, 3, false>(a, 7.0f);
    else if constexpr (FMT == MO_EF_E1M2) return round_minifloat<2, 1, false>(a, 3.5f);
    else if constexpr (FMT == MO_EF_E3M0) return round_minifloat<0, -2, true>(a, 16.0f);
    else if constexpr (FMT == MO_EF_E2M1) return round_minifloat<1, 0, false>(a, 6.0f);
    else if constexpr (FMT == MO_EF_E3M2) return round_minifloat<2, -2, false>(a, 28.0f);
    else return round_minifloat<3, 0, false>(a, 7.5f);  // E2M3
}

__device__ __forceinline__ float convert_runtime(float a, int fmt) {
    switch (fmt) {
        case MO_EF_E4M3: return convert_elem<MO_EF_E4M3>(a);
        case MO_EF_E5M2: return convert_elem<MO_EF_E5M2>(a);
        case MO_EF_INT8: return convert_elem<MO_EF_INT8>(a);
        case MO_EF_E0M3: return convert_elem<MO_EF_E0M3>(a);
        case MO_EF_E1M2: return convert_elem<MO_EF_E1M2>(a);
        case MO_EF_E3M0: return convert_elem<MO_EF_E3M0>(a);
        case MO_EF_E2M1: return convert_elem<MO_EF_E2M1>(a);
        case MO_EF_E3M2: return convert_elem<MO_EF_E3M2>(a);
        default: return convert_elem<MO_EF_E2M3>(a);
    }
}

__host__ __device__ __forceinline__ float elem_format_max(int fmt) {
    switch (fmt) {
        case MO_EF_E4M3: return 448.0f;
        case MO_EF_E5M2: return 57344.0f;
        case MO_EF_INT8: return 127.0f;
        case MO_EF_E0M3: return 7.0f;
        case MO_EF_E1M2: return 3.5f;
        case MO_EF_E3M0: return 16.0f;
        case MO_EF_E2M1: return 6.0f;
        case MO_EF_E3M2: return 28.0f;
        default: return 7.5f;
    }
}

struct BlockScale { float scale, unscale; };

// amax: block abs-max with |x| clamped to FLT_MAX and NaN elements ignored.
template <int FMT>
__device__ __forceinline__ BlockScale block_scale(float amax, int scale_fmt, bool has_global,
                                                  float global_amax) {
    BlockScale s = {1.0f, 1.0f};
    if (amax == 0.0f) return s;  // finite by construction
    const float fmax = elem_format_max(FMT);
    if (has_global) {
        // two-level scale: the block's unscale, quantised to scale_fmt relative to the global amax
        if (global_amax == 0.0f || !(__builtin_fabsf(global_amax) < __builtin_inff())) return s;
        const float smax = elem_format_max(scale_fmt);
        const float local_unscale = amax / fmax;
        const double two_level = (double)smax * (double)(fmax / global_amax);
        const double q = (double)convert_runtime((float)((double)local_unscale * two_level), scale_fmt) /
                         two_level;
        s.scale = (float)(1.0 / q);
        s.unscale = (float)q;
    } else if (scale_fmt == MO_EF_E8M0) {
        // unscale = 2^ceil(log2(amax / fmax)), read off the bits of the fp32 quotient
        const uint32_t bits = f2u(amax / fmax), ef = (bits >> 23) & 0xFFu, mant = bits & 0x7FFFFFu;
        const int e = (mant > 0 && ef != 0xFEu && !(ef == 0 && mant <= 0x400000u)) ? (int)ef - 126
                                                                                   : (int)ef - 127;
        s.scale = __builtin_ldexpf(1.0f, -e);
        s.unscale = __builtin_ldexpf(1.0f, e);
    } else {
        const double sc = (double)fmax / (double)amax;
        const double inv = (double)convert_runtime((float)(1.0 / sc), scale_fmt);
        s.scale = (float)(1.0 / inv);
        s.unscale = (float)inv;
    }
    return s;
}

// One chunk of 8 elements under the scale of its block.
template <int FMT>
__device__ __forceinline__ void block_fp_chunk(const float (&v)[8], const BlockScale& s, float (&o)[8]) {
    if constexpr (FMT == MO_EF_E4M3) {   // two elements per conversion each way
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
            float a = __builtin_fabsf(v[j]) * s.scale, b = __builtin_fabsf(v[j + 1]) * s.scale;
            a = a > 448.0f ? 448.0f : a;   // NaN stays NaN
            b = b > 448.0f ? 448.0f : b;
            round_e4m3_pair<false>(a, b);
            o[j] = a * s.unscale;
            o[j + 1] = b * s.unscale;
        }
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = convert_elem<FMT>(__builtin_fabsf(v[j]) * s.scale) * s.unscale;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = v[j] < 0.0f ? -o[j] : o[j];
}

// The lane's share of a block abs-max: NaN elements dropped, infinities clamped to FLT_MAX.
__device__ __forceinline__ uint32_t block_fp_absmax(const float (&v)[8]) {
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        uint32_t t = f2u(v[j]) & 0x7FFFFFFFu;
        t = t > 0x7F800000u ? 0u : (t < 0x7F7FFFFFu ? t : 0x7F7FFFFFu);
        m = t > m ? t : m;
    }
    return m;
}

}  // namespace mo
