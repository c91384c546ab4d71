// What the gradient kernels share: products of 16-bit operands on the matrix cores, operands turned on their way out of
// LDS, results rounded two to a word, tiles spread over the XCDs.
#pragma once

#include "common.h"

namespace mo {

typedef float f32x16 __attribute__((ext_vector_type(16)));

// 16 products for each of 32 x 32 sums; a lane holds 8 of the 16 of one row (a) and of one column (b)
template <int DT>
__device__ __forceinline__ f32x16 mfma_32x32x16(u32x4 a, u32x4 b, f32x16 c) {
    typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
    typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
    if constexpr (DT == MO_BF16) {
        bf16x8 av, bv;
        __builtin_memcpy(&av, &a, 16);
        __builtin_memcpy(&bv, &b, 16);
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bv, c, 0, 0, 0);
    } else {
        f16x8 av, bv;
        __builtin_memcpy(&av, &a, 16);
        __builtin_memcpy(&bv, &b, 16);
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bv, c, 0, 0, 0);
    }
}

// Two results as one word of their type
template <int DT>
__device__ __forceinline__ uint32_t round_pair(float lo, float hi) {
    if constexpr (DT == MO_BF16) return f32x2_to_bf16x2(lo, hi);
    else return f32_to_f16_bits(lo) | (f32_to_f16_bits(hi) << 16);
}

// ds_read_b64_tr_b16: 16 lanes read 4 rows of 16 columns, each lane gets 4 rows of one
__device__ __forceinline__ u32x2 lds_transposed(const uint8_t* p) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p);
    u32x2 r;
    __builtin_memcpy(&r, &v, 8);
    return r;
}

// Workgroups go round the eight XCDs: the tile of `total` that this one takes, so that each XCD gets a run of tiles
__device__ __forceinline__ uint32_t xcd_tile(uint32_t total) {
    const uint32_t xcd = blockIdx.x & 7u, q = total >> 3, rest = total & 7u;
    return xcd * q + (xcd < rest ? xcd : rest) + (blockIdx.x >> 3);
}

}  // namespace mo
