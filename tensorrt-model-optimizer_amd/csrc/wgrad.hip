// Weight gradient of a linear layer behind a fake-quantised weight, for gfx950:
//
//   dw[n, k] = |w[n, k]| <= amax(n, k) ? T(sum over t of dy[t, n] * x[t, k]) : 0
//
// the product of the library's GEMM and the mask of ste.hip in one pass.  A training step has a few
// hundred tokens, so the contraction is short and the [N, K] result is what costs: the two launches
// write it, read it back with the weight and write it again.
//
// Both operands are contiguous along the dimension that is kept and strided along the one that is summed,
// the opposite of what the matrix instructions read.  A lane therefore loads the same 8 columns of 8
// tokens (8 accesses of 16 bytes, 256 contiguous bytes a row), turns them in registers with one byte
// permutation per two elements and stores 8 columns of 8 tokens to LDS.  A column is a row of 64 tokens
// there, its eight 16-byte slots permuted so that neither the stores (columns 8 apart) nor the operand
// reads (adjacent columns) conflict.  128 x 128 results a workgroup
// of four wavefronts, 64 x 64 each in 64 accumulators; the loads of the next 64 tokens are in
// flight during the matrix instructions, and three workgroups a compute unit overlap the
// stores of one with the products of another.  The result goes through LDS once more, so that the weight
// is read and the gradient written in rows of 256 bytes.
//
// Measured on a 14336 x 4096 bf16 weight with an amax a row, against the library's product and mo_ste_mask: 64
// tokens 44 us (89) = 5.3 TB/s of weight and gradient, 256 tokens 67 (109), 512 tokens 96 (140) = 0.62
// PFLOP/s, 1024 tokens 179 (200).  Up to some 100 tokens memory bounds it, beyond that the loads of the
// operands: 96 KB in flight a compute unit (128 bytes a lane), a quarter of them past L2.  More than three wavefronts a
// SIMD do not fit the registers (128 of them spill: 243 us at 512 tokens).
// Sums run in fp32 over the tokens in order, 16 an instruction, and round once: against sums in 64 bits as many results
// are off by a rounding as the library's product has (32 to 1024 tokens, both types: the same ones).
#include "common.h"

namespace mo {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int kWgTile = 128;     // results of a workgroup along n and along k
constexpr int kWgTokens = 64;    // tokens of a step
constexpr int kWgGroup = 8;      // n tiles that the workgroups of one XCD share their k tiles over

template <int DT>
__device__ __forceinline__ f32x16 wgrad_mfma(u32x4 a, u32x4 b, f32x16 c) {
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

template <int DT>
__device__ __forceinline__ uint32_t wgrad_pair(float lo, float hi) {
    if constexpr (DT == MO_BF16) return f32x2_to_bf16x2(lo, hi);
    else return f32_to_f16_bits(lo) | (f32_to_f16_bits(hi) << 16);
}

// Byte offset of a column's octet of tokens in its operand tile.  A 16-byte store is served eight lanes at a
// time, in order: the same column of eight chunks here, eight different slots.  A 16-byte read is served
// sixteen lanes at a time, lanes 0 - 3, 12 - 15 and 20 - 27, then 4 - 11, 16 - 19 and 28 - 31, and so for the upper
// half (measured lane by lane): their even columns, and their odd ones, have eight different slots.
__device__ __forceinline__ int wgrad_slot(int col, int octet) {
    return col * (kWgTokens * 2) + ((octet ^ col ^ (col >> 3)) & 7) * 16;
}

// 8 columns of 8 tokens of the step at t (uniform); p: the first of them in that step.  Tokens past the end
// are zero in both operands.
__device__ __forceinline__ void wgrad_load(const uint16_t* __restrict__ p, int64_t width, int64_t t, int octet,
                                           int64_t tokens, u32x4 (&r)[8]) {
    if (t + kWgTokens <= tokens) {
#pragma unroll
        for (int i = 0; i < 8; ++i) r[i] = *(const u32x4*)(p + i * width);
    } else {
        const int left = (int)(tokens - t) - octet * 8;   // of this octet, at most 0 past the end
        const u32x4 zero = {0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            r[i] = zero;
            if (i < left) r[i] = *(const u32x4*)(p + i * width);
        }
    }
}

template <int DT>
__global__ __launch_bounds__(256, 3) void wgrad_masked_kernel(
    const uint16_t* __restrict__ dy, const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
    uint16_t* __restrict__ dw, int64_t tokens, int64_t n_all, int64_t k_all, uint32_t tiles_n, uint32_t tiles_k,
    const void* __restrict__ amax, int amax_dtype, uint32_t inner, int narrow) {
    __shared__ __align__(16) uint8_t lds[2 * kWgTile * kWgTokens * 2];
    uint8_t* const xs = lds;                               // columns of x: [128][64 tokens]
    uint8_t* const ys = lds + kWgTile * kWgTokens * 2;     // columns of dy

    // workgroups go round the eight XCDs: each XCD gets a run of tiles, group by group of n tiles with the
    // k tiles outside, so that what runs at a time shares its operands in the XCD's L2
    const uint32_t total = tiles_n * tiles_k, xcd = blockIdx.x & 7u, q = total >> 3, rest = total & 7u;
    const uint32_t id = xcd * q + (xcd < rest ? xcd : rest) + (blockIdx.x >> 3);
    const uint32_t per_group = kWgGroup * tiles_k, group = id / per_group, first = group * kWgGroup;
    const uint32_t wide = tiles_n - first < kWgGroup ? tiles_n - first : kWgGroup;
    const uint32_t in_group = id - group * per_group;
    const int64_t n0 = (int64_t)(first + in_group % wide) * kWgTile, k0 = (int64_t)(in_group / wide) * kWgTile;

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // loading: lanes 0 .. 127 x, 128 .. 255 dy; 16 chunks of 8 columns by 8 octets of tokens
    const bool loads_y = threadIdx.x >= 128;
    const int chunk = threadIdx.x & 15, octet = (threadIdx.x >> 4) & 7;
    const int64_t width = loads_y ? n_all : k_all;
    int64_t col = (loads_y ? n0 : k0) + chunk * 8;
    col = col < width ? col : width - 8;                   // past the edge: results that are not stored
    const uint16_t* src = (loads_y ? dy : x) + octet * 8 * width + col;
    uint8_t* const dst = loads_y ? ys : xs;

    // multiplying: 64 x 64 of a wavefront, 2 x 2 blocks of 32
    const int wk = (wave & 1) * 64, wn = (wave >> 1) * 64, l32 = lane & 31, half = lane >> 5;
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    u32x4 r[8];
    wgrad_load(src, width, 0, octet, tokens, r);
    for (int64_t t = 0; t < tokens; t += kWgTokens) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            u32x4 o;
#pragma unroll
            for (int p = 0; p < 4; ++p)
                o[p] = __builtin_amdgcn_perm(r[2 * p + 1][j >> 1], r[2 * p][j >> 1], (j & 1) ? 0x07060302u : 0x05040100u);
            *(u32x4*)(dst + wgrad_slot(chunk * 8 + j, octet)) = o;
        }
        __syncthreads();
        src += kWgTokens * width;
        if (t + kWgTokens < tokens) wgrad_load(src, width, t + kWgTokens, octet, tokens, r);
#pragma unroll
        for (int s = 0; s < kWgTokens / 16; ++s) {
            u32x4 a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                a[i] = *(const u32x4*)(xs + wgrad_slot(wk + i * 32 + l32, 2 * s + half));
                b[i] = *(const u32x4*)(ys + wgrad_slot(wn + i * 32 + l32, 2 * s + half));
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = wgrad_mfma<DT>(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }

    // the weight's chunks of this lane, 8 rows 16 apart; loaded before the results go through LDS
    RawChunk<DT> rw[8];
    uint32_t raw_limit[8];
    const int out_chunk = threadIdx.x & 15, out_row = threadIdx.x >> 4;
    int64_t k = k0 + out_chunk * 8;
    const bool k_ok = k < k_all;
    k = k_ok ? k : k_all - 8;
    // inner elements share an amax and a row is a whole number of them; 0: one amax
    const int64_t amax_row = inner ? (uint32_t)k_all / inner : 0, amax_col = inner ? (uint32_t)k / inner : 0;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        int64_t n = n0 + u * 16 + out_row;
        n = n < n_all ? n : n_all - 1;
        load_raw<DT>(w, n * k_all + k, rw[u]);
    }
    // the limits as fp32 bits, one branch for all of them
    auto limits = [&](auto read) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            int64_t n = n0 + u * 16 + out_row;
            n = n < n_all ? n : n_all - 1;
            raw_limit[u] = read(n * amax_row + amax_col);
        }
    };
    if (amax_dtype == MO_F32) limits([&](int64_t i) { return ((const uint32_t*)amax)[i]; });
    else if (amax_dtype == MO_BF16) limits([&](int64_t i) { return (uint32_t)((const uint16_t*)amax)[i] << 16; });
    else limits([&](int64_t i) { return f2u(f16_bits_to_f32(((const uint16_t*)amax)[i])); });
    // 16-byte slots of a row of 128 results, permuted by the row number
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                // accumulators 4 g .. 4 g + 3 of lane l: k = 8 g + 4 (l / 32) + 0 .. 3, n = l % 32
                const int row = wn + j * 32 + l32, slot = (wk + i * 32) / 8 + g;
                u32x2 o;
                o.x = wgrad_pair<DT>(acc[i][j][4 * g], acc[i][j][4 * g + 1]);
                o.y = wgrad_pair<DT>(acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]);
                *(u32x2*)(lds + row * 256 + ((slot ^ row) & 15) * 16 + half * 8) = o;
            }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int row = u * 16 + out_row;
        u32x4 g = *(const u32x4*)(lds + row * 256 + ((out_chunk ^ row) & 15) * 16);
        float v[8], limit = u2f(raw_limit[u]);
        const float rounded = DT == MO_BF16 ? round_to_bf16(limit) : f16_bits_to_f32(f32_to_f16_bits(limit));
        limit = narrow ? rounded : limit;
        unpack_raw<DT>(rw[u], v);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            g[j] &= (__builtin_fabsf(v[2 * j]) <= limit ? 0x0000FFFFu : 0u) |
                    (__builtin_fabsf(v[2 * j + 1]) <= limit ? 0xFFFF0000u : 0u);
        if (k_ok && n0 + row < n_all) __builtin_nontemporal_store(g, (u32x4*)(dw + (n0 + row) * k_all + k));
    }
}

}  // namespace mo

extern "C" int mo_wgrad_masked(const void* dy, const void* x, const void* w, void* dw, int64_t tokens, int64_t n,
                               int64_t k, int dtype, const void* amax, int amax_dtype, int64_t inner,
                               int narrow_amax, void* stream) {
    if (tokens <= 0 || n < 0 || k < 0 || inner < 0) return MO_ERR_ARG;
    if (dtype < MO_F32 || dtype > MO_BF16 || amax_dtype < MO_F32 || amax_dtype > MO_BF16) return MO_ERR_DTYPE;
    if (dtype == MO_F32) return MO_ERR_UNSUPPORTED;
    if (n == 0 || k == 0) return MO_OK;
    if (!dy || !x || !w || !dw || !amax) return MO_ERR_ARG;
    if (n % 8 || k % 8 || inner % 8 || (inner && k % inner) || k > 0x7FFFFFFF || (((uintptr_t)dy | (uintptr_t)x | (uintptr_t)w | (uintptr_t)dw) & 15u))
        return MO_ERR_UNSUPPORTED;
    const int64_t tn = (n + mo::kWgTile - 1) / mo::kWgTile, tk = (k + mo::kWgTile - 1) / mo::kWgTile;
    if (tn > 0x3FFFFFFF / mo::kWgGroup || tk > 0x3FFFFFFF / mo::kWgGroup || tn * tk > 0x7FFFFFFF) return MO_ERR_UNSUPPORTED;
    hipStream_t s = (hipStream_t)stream;
#define CALL(DT)                                                                                            \
    mo::wgrad_masked_kernel<DT><<<(unsigned)(tn * tk), 256, 0, s>>>(                                        \
        (const uint16_t*)dy, (const uint16_t*)x, (const uint16_t*)w, (uint16_t*)dw, tokens, n, k, (uint32_t)tn, \
        (uint32_t)tk, amax, amax_dtype, (uint32_t)inner, narrow_amax)
    if (dtype == MO_BF16) CALL(MO_BF16); else CALL(MO_F16);
#undef CALL
    return hipGetLastError() == hipSuccess ? MO_OK : MO_ERR_LAUNCH;
}
