// Backward of the fake quantisers for gfx950: the straight-through estimator that lets a gradient
// through where the input lay inside the quantisation range and stops it elsewhere.
//
//   dx[i] = |x[i]| <= amax(i) ? dy[i] : 0          (a NaN on either side of the comparison stops it)
//
// HBM-bound: x and dy are read once and dx is written once, 6 bytes per bf16 element.  The gradient
// is moved as bits, so its values (NaN payloads, -0) pass unchanged.  One workgroup per tile of
// 1024 chunks of 8 elements, four chunks of x and four of dy in flight per lane ahead of the
// first store, as in the forward kernels.
// Measured on a 14336 x 4096 bf16 weight with one amax per row: 58 us = 6.0 TB/s, where the absolute
// value, the comparison and the selection as three tensor operations took 163 us; no occupancy cap
// helps (58 us from none to 36 KB of unused LDS, 61 with 48 KB).
#include "common.h"

namespace mo {

enum { STE_TENSOR = 0, STE_CHUNK = 1 };

constexpr int kSteU = 4;
constexpr int kSteTileChunks = 256 * kSteU;

// amax as the comparison sees it.  `narrow`: the amax is a 0-dim tensor of another type, which the
// comparison converts to the type of x first.
template <int DT>
__device__ __forceinline__ float ste_limit(const void* amax, int amax_dtype, int64_t i, int narrow) {
    const float a = load_scalar(amax, amax_dtype, i);
    if (!narrow) return a;
    if constexpr (DT == MO_BF16) return round_to_bf16(a);
    else if constexpr (DT == MO_F16) return f16_bits_to_f32(f32_to_f16_bits(a));
    else return a;
}

template <int DT>
__device__ __forceinline__ void ste_select(const RawChunk<DT>& rx, RawChunk<DT>& rg, float limit) {
    float v[8];
    unpack_raw<DT>(rx, v);
    if constexpr (DT == MO_F32) {
        uint32_t w[8] = {rg.a.x, rg.a.y, rg.a.z, rg.a.w, rg.b.x, rg.b.y, rg.b.z, rg.b.w};
#pragma unroll
        for (int j = 0; j < 8; ++j) w[j] = __builtin_fabsf(v[j]) <= limit ? w[j] : 0u;
        rg.a = u32x4{w[0], w[1], w[2], w[3]};
        rg.b = u32x4{w[4], w[5], w[6], w[7]};
    } else {
        uint32_t w[4] = {rg.a.x, rg.a.y, rg.a.z, rg.a.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t keep = (__builtin_fabsf(v[2 * j]) <= limit ? 0x0000FFFFu : 0u) |
                                  (__builtin_fabsf(v[2 * j + 1]) <= limit ? 0xFFFF0000u : 0u);
            w[j] &= keep;
        }
        rg.a = u32x4{w[0], w[1], w[2], w[3]};
    }
}

template <int DT>
__device__ __forceinline__ void store_raw(void* p, int64_t i, const RawChunk<DT>& r) {
    if constexpr (DT == MO_F32) {
        u32x4* q = (u32x4*)((float*)p + i);
        __builtin_nontemporal_store(r.a, q);
        __builtin_nontemporal_store(r.b, q + 1);
    } else {
        __builtin_nontemporal_store(r.a, (u32x4*)((uint16_t*)p + i));
    }
}

template <int DT>
__device__ __forceinline__ void ste_elem(const void* x, const void* dy, void* dx, int64_t i, float limit) {
    const bool keep = __builtin_fabsf(load_elem<DT>(x, i)) <= limit;
    if constexpr (DT == MO_F32) ((uint32_t*)dx)[i] = keep ? ((const uint32_t*)dy)[i] : 0u;
    else ((uint16_t*)dx)[i] = keep ? ((const uint16_t*)dy)[i] : (uint16_t)0;
}

// x viewed as [outer, axis, inner]: TENSOR one amax, CHUNK inner % 8 == 0 (a chunk shares its amax)
template <int DT, int KIND>
__global__ __launch_bounds__(256) void ste_mask_kernel(const void* __restrict__ x,
                                                       const void* __restrict__ dy,
                                                       void* __restrict__ dx, int64_t n, int64_t axis,
                                                       int64_t inner, const void* __restrict__ amax,
                                                       int amax_dtype, int narrow) {
    const int64_t chunks = n >> 3;
    const int64_t c0 = (int64_t)blockIdx.x * kSteTileChunks + threadIdx.x;
    if (chunks > 0) {
        const int64_t inner_chunks = KIND == STE_CHUNK ? inner >> 3 : 1;
        RawChunk<DT> rx[kSteU], rg[kSteU];
        float lim[kSteU];
#pragma unroll
        for (int u = 0; u < kSteU; ++u) {
            int64_t c = c0 + u * 256;
            c = c < chunks ? c : chunks - 1;
            load_raw<DT>(x, c << 3, rx[u]);
            load_raw<DT>(dy, c << 3, rg[u]);
            int64_t a = 0;
            if constexpr (KIND == STE_CHUNK) {
                if (chunks <= 0xFFFFFFFFll) a = (uint32_t)c / (uint32_t)inner_chunks;
                else a = c / inner_chunks;
                a = a < axis ? a : a % axis;
            }
            lim[u] = ste_limit<DT>(amax, amax_dtype, a, narrow);
        }
#pragma unroll
        for (int u = 0; u < kSteU; ++u) {
            const int64_t c = c0 + u * 256;
            ste_select<DT>(rx[u], rg[u], lim[u]);
            if (c < chunks) store_raw<DT>(dx, c << 3, rg[u]);
        }
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x < (n & 7)) {   // the last n % 8 elements
        const int64_t i = (chunks << 3) + threadIdx.x;
        const int64_t a = KIND == STE_TENSOR ? 0 : (i / inner) % axis;
        ste_elem<DT>(x, dy, dx, i, ste_limit<DT>(amax, amax_dtype, a, narrow));
    }
}

// Any layout and any alignment, one element at a time.
template <int DT>
__global__ __launch_bounds__(256) void ste_mask_elem_kernel(const void* __restrict__ x,
                                                            const void* __restrict__ dy,
                                                            void* __restrict__ dx, int64_t n,
                                                            int64_t axis, int64_t inner,
                                                            const void* __restrict__ amax,
                                                            int amax_dtype, int narrow) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        ste_elem<DT>(x, dy, dx, i, ste_limit<DT>(amax, amax_dtype, (i / inner) % axis, narrow));
}

template <int DT>
static int launch_ste(const void* x, const void* dy, void* dx, int64_t outer, int64_t axis, int64_t inner,
                      const void* amax, int amax_dtype, int narrow, hipStream_t s) {
    const int64_t n = outer * axis * inner;
    const bool aligned = (((uintptr_t)x | (uintptr_t)dy | (uintptr_t)dx) & 15u) == 0;
    int64_t tiles = ((n >> 3) + kSteTileChunks - 1) / kSteTileChunks;
    if (tiles < 1) tiles = 1;
    if (aligned && (axis == 1 || inner % 8 == 0) && tiles <= 0x7FFFFFFF) {
        if (axis == 1)
            ste_mask_kernel<DT, STE_TENSOR><<<(unsigned)tiles, 256, 0, s>>>(x, dy, dx, n, axis, inner, amax, amax_dtype, narrow);
        else
            ste_mask_kernel<DT, STE_CHUNK><<<(unsigned)tiles, 256, 0, s>>>(x, dy, dx, n, axis, inner, amax, amax_dtype, narrow);
        return MO_OK;
    }
    int64_t b = (n + 255) / 256;
    if (b > 16384) b = 16384;
    ste_mask_elem_kernel<DT><<<(unsigned)b, 256, 0, s>>>(x, dy, dx, n, axis, inner, amax, amax_dtype, narrow);
    return MO_OK;
}

}  // namespace mo

extern "C" int mo_ste_mask(const void* x, const void* dy, void* dx, int64_t outer, int64_t axis,
                           int64_t inner, int dtype, const void* amax, int amax_dtype,
                           int narrow_amax, void* stream) {
    if (outer < 0 || axis < 0 || inner < 0) return MO_ERR_ARG;
    if (dtype < MO_F32 || dtype > MO_BF16 || amax_dtype < MO_F32 || amax_dtype > MO_BF16) return MO_ERR_DTYPE;
    if (outer == 0 || axis == 0 || inner == 0) return MO_OK;
    if (!x || !dy || !dx || !amax) return MO_ERR_ARG;
    hipStream_t s = (hipStream_t)stream;
    int rc;
    switch (dtype) {
        case MO_F32: rc = mo::launch_ste<MO_F32>(x, dy, dx, outer, axis, inner, amax, amax_dtype, narrow_amax, s); break;
        case MO_F16: rc = mo::launch_ste<MO_F16>(x, dy, dx, outer, axis, inner, amax, amax_dtype, narrow_amax, s); break;
        default: rc = mo::launch_ste<MO_BF16>(x, dy, dx, outer, axis, inner, amax, amax_dtype, narrow_amax, s); break;
    }
    if (rc != MO_OK) return rc;
    return hipGetLastError() == hipSuccess ? MO_OK : MO_ERR_LAUNCH;
}
