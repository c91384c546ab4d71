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
// tokens 44 us (89) = 5.3 TB/s of weight and gradient, 256 tokens 67 (109), 512 tokens 96 (140), 1024 tokens 160 (200); from 384
// tokens on the kernel further below takes over.  Up to some 100 tokens memory bounds it, beyond that the loads of the
// operands: 96 KB in flight a compute unit (128 bytes a lane), a quarter of them past L2.  More than three wavefronts a
// SIMD do not fit the registers (128 of them spill: 243 us at 512 tokens).
// Sums run in fp32 over the tokens in order, 16 an instruction, and round once: against sums in 64 bits as many results
// are off by a rounding as the library's product has (32 to 1024 tokens, both types: the same ones).
#include "mfma_ops.h"

namespace mo {

constexpr int kWgTile = 128;     // results of a workgroup along n and along k
constexpr int kWgTokens = 64;    // tokens of a step
constexpr int kWgLongTokens = 32;   // the same of the kernel for many tokens
constexpr int kWgGroup = 8;      // n tiles that the workgroups of one XCD share their k tiles over

// First result of this workgroup along n and along k: each XCD gets a run of tiles, group by group of n tiles with the
// k tiles outside, so that what runs at a time shares its operands in the XCD's L2
struct WgradOrigin { int64_t n, k; };
__device__ __forceinline__ WgradOrigin wgrad_origin(uint32_t tiles_n, uint32_t tiles_k) {
    const uint32_t id = xcd_tile(tiles_n * tiles_k);
    const uint32_t per_group = kWgGroup * tiles_k, group = id / per_group, first = group * kWgGroup;
    const uint32_t wide = tiles_n - first < kWgGroup ? tiles_n - first : kWgGroup;
    const uint32_t in_group = id - group * per_group;
    return {(int64_t)(first + in_group % wide) * kWgTile, (int64_t)(in_group / wide) * kWgTile};
}

// The weight's chunks of a lane at column k, 8 rows 16 apart from n on, and their limits as fp32 bits (one branch for all of them).
// `inner` elements share an amax and a row is a whole number of them; 0: one amax
template <int DT>
__device__ __forceinline__ void wgrad_weight(const uint16_t* __restrict__ w, int64_t n_first, int64_t n_all, int64_t k, int64_t k_all,
                                             const void* __restrict__ amax, int amax_dtype, uint32_t inner,
                                             RawChunk<DT> (&rw)[8], uint32_t (&raw_limit)[8]) {
    const int64_t amax_row = inner ? (uint32_t)k_all / inner : 0, amax_col = inner ? (uint32_t)k / inner : 0;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        int64_t n = n_first + u * 16;
        n = n < n_all ? n : n_all - 1;
        load_raw<DT>(w, n * k_all + k, rw[u]);
    }
    auto limits = [&](auto read) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            int64_t n = n_first + u * 16;
            n = n < n_all ? n : n_all - 1;
            raw_limit[u] = read(n * amax_row + amax_col);
        }
    };
    if (amax_dtype == MO_F32) limits([&](int64_t i) { return ((const uint32_t*)amax)[i]; });
    else if (amax_dtype == MO_BF16) limits([&](int64_t i) { return (uint32_t)((const uint16_t*)amax)[i] << 16; });
    else limits([&](int64_t i) { return f2u(f16_bits_to_f32(((const uint16_t*)amax)[i])); });
}

// The sums of a wavefront at wn, wk of the tile, rounded, to LDS: 16-byte slots of a row of 128 results, permuted by the
// row number
template <int DT>
__device__ __forceinline__ void wgrad_results(uint8_t* lds, const f32x16 (&acc)[2][2], int wn, int wk, int lane) {
    const int l32 = lane & 31, half = lane >> 5;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                // accumulators 4 g .. 4 g + 3 of lane l: k = 8 g + 4 (l / 32) + 0 .. 3, n = l % 32
                const int row = wn + j * 32 + l32, slot = (wk + i * 32) / 8 + g;
                u32x2 o;
                o.x = round_pair<DT>(acc[i][j][4 * g], acc[i][j][4 * g + 1]);
                o.y = round_pair<DT>(acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]);
                *(u32x2*)(lds + row * 256 + ((slot ^ row) & 15) * 16 + half * 8) = o;
            }
}
// 8 results of a row of the tile
__device__ __forceinline__ u32x4 wgrad_result(const uint8_t* lds, int row, int chunk) {
    return *(const u32x4*)(lds + row * 256 + ((chunk ^ row) & 15) * 16);
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

    const WgradOrigin origin = wgrad_origin(tiles_n, tiles_k);
    const int64_t n0 = origin.n, k0 = origin.k;

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
                for (int j = 0; j < 2; ++j) acc[i][j] = mfma_32x32x16<DT>(a[i], b[j], acc[i][j]);
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
    wgrad_weight<DT>(w, n0 + out_row, n_all, k, k_all, amax, amax_dtype, inner, rw, raw_limit);
    wgrad_results<DT>(lds, acc, wn, wk, lane);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int row = u * 16 + out_row;
        u32x4 g = wgrad_result(lds, row, out_chunk);
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

// ------------------------------------------------------------------------------ many tokens
// The same with the operands in LDS as they lie in memory, [token][column], and turned on the way out of it
// (ds_read_b64_tr_b16: 16 lanes read 4 tokens of 16 columns, each lane gets 4 tokens of one), which leaves out the byte
// permutations.  32 tokens a step, three LDS stages: one is multiplied, the next is complete, so that the first operands of a
// step are read before its only barrier, and the loads of the one after that are written to LDS between the products; global
// loads run two steps further ahead, in registers.  The weight is read first and kept as a bit an element; the
// same products in the same order, the same bits.  bf16: 1024 tokens x 14336 x 4096 160 -> 139 us, x 4096 x 4096 55.7 -> 45.5,
// 512 tokens 94 -> 88 and 35 -> 30.5; at 256 62 and 62, 26 and 25, at 64, where memory bounds both and the early
// weight only lengthens a workgroup, 44 and 47.  Tried on it without gain: the weight read in quarters between the steps,
// workgroups of a compute unit started apart.
// Byte offset of 8 columns of a token in its operand tile (256 bytes a token).  A transposed read takes 4 tokens of 64
// bytes for 32 lanes: the four lie in different quarters of a row.
__device__ __forceinline__ int wgrad_row_slot(int token, int octet) {
    return token * 256 + ((octet ^ (token << 2)) & 15) * 16;
}

// The mask on the two elements of a word at a time: |w| <= amax is an order of the 15 bits below the sign, with amax
// rounded down to the type.  0x8000 + amax - |w| has its top bit where the element is kept and never borrows from the other
// half; an amax that lets nothing through (a NaN, a negative one) is one below zero.
template <int DT>
__device__ __forceinline__ uint32_t wgrad_limit(float amax, int narrow) {
    uint32_t bits;
    if constexpr (DT == MO_BF16) {
        if (narrow) amax = round_to_bf16(amax);
        bits = (f2u(amax) >> 16) & 0x7FFFu;
    } else {
        if (narrow) amax = f16_bits_to_f32(f32_to_f16_bits(amax));
        bits = f32_to_f16_bits(__builtin_fabsf(amax)) & 0x7FFFu;
        if (f16_bits_to_f32(bits) > __builtin_fabsf(amax)) --bits;
    }
    bits = amax >= 0.0f ? 0x8000u + bits : 0x7FFFu;
    return bits | bits << 16;
}
// The bits of 16 words, the first at 0 and 16
__device__ __forceinline__ void wgrad_keep(uint32_t& bits, uint32_t w, uint32_t limit) {
    bits = (bits >> 1) | ((limit - (w & 0x7FFF7FFFu)) & 0x80008000u);
}
// All bits of a half whose lowest bit is set
__device__ __forceinline__ uint32_t wgrad_mask(uint32_t bits) { return (bits & 0x00010001u) * 0xFFFFu; }

template <int DT>
__global__ __launch_bounds__(256, 3) void wgrad_masked_long_kernel(
    const uint16_t* __restrict__ dy, const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
    uint16_t* __restrict__ dw, int64_t tokens, int64_t n_all, int64_t k_all, uint32_t tiles_n, uint32_t tiles_k,
    const void* __restrict__ amax, int amax_dtype, uint32_t inner, int narrow) {
    constexpr int kTile = kWgLongTokens * 256, kStage = 2 * kTile, kChunks = kWgLongTokens / 16;
    __shared__ __align__(16) uint8_t lds[3 * kStage];   // a stage: x, then dy

    const WgradOrigin origin = wgrad_origin(tiles_n, tiles_k);
    const int64_t n0 = origin.n, k0 = origin.k;

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // Buffer descriptors of one step's rows (scalar): what is past the last token reads as zero, what is past the
    // edge of a row belongs to results that are not stored
    const int chunk = threadIdx.x & 15, token0 = threadIdx.x >> 4;
    const uint32_t x_row = (uint32_t)k_all * 2, y_row = (uint32_t)n_all * 2;
    const uint16_t *x_at = x, *y_at = dy;
    int64_t left = tokens;
    uint32_t x_off[kChunks], y_off[kChunks];
    int dst[kChunks];
#pragma unroll
    for (int i = 0; i < kChunks; ++i) {
        const int token = token0 + i * 16;
        x_off[i] = (uint32_t)token * x_row + (uint32_t)(k0 + chunk * 8) * 2;
        y_off[i] = (uint32_t)token * y_row + (uint32_t)(n0 + chunk * 8) * 2;
        dst[i] = wgrad_row_slot(token, chunk);
    }
    struct Stage { u32x4 x[kChunks], y[kChunks]; };
    auto load = [&](Stage& r) {
        const uint32_t rows = (uint32_t)(left < 0 ? 0 : left < kWgLongTokens ? left : kWgLongTokens);
        const auto x_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)x_at, 0, (int)(rows * x_row), 0x00020000);
        const auto y_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)y_at, 0, (int)(rows * y_row), 0x00020000);
#pragma unroll
        for (int i = 0; i < kChunks; ++i) {
            r.x[i] = __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, x_off[i], 0, 0);
            r.y[i] = __builtin_amdgcn_raw_buffer_load_b128(y_rsrc, y_off[i], 0, 0);
        }
        x_at += kWgLongTokens * k_all;
        y_at += kWgLongTokens * n_all;
        left -= kWgLongTokens;
    };
    auto store_x = [&](const Stage& r, int at) {
#pragma unroll
        for (int i = 0; i < kChunks; ++i) *(u32x4*)(lds + at + dst[i]) = r.x[i];
    };
    auto store_y = [&](const Stage& r, int at) {
#pragma unroll
        for (int i = 0; i < kChunks; ++i) *(u32x4*)(lds + at + kTile + dst[i]) = r.y[i];
    };
    Stage r0, r1;

    // What the mask keeps of this lane's results, 8 chunks of rows 16 apart: a bit an element, made before the sums
    // need the registers
    uint32_t keep[2] = {0, 0};
    const int out_chunk = threadIdx.x & 15, out_row = threadIdx.x >> 4;
    int64_t k = k0 + out_chunk * 8;
    const bool k_ok = k < k_all;
    k = k_ok ? k : k_all - 8;
    {
        RawChunk<DT> rw[8];
        uint32_t raw_limit[8];
        wgrad_weight<DT>(w, n0 + out_row, n_all, k, k_all, amax, amax_dtype, inner, rw, raw_limit);
        load(r0);
        load(r1);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const uint32_t limit = wgrad_limit<DT>(u2f(raw_limit[u]), narrow);
            const u32x4 words = rw[u].a;
#pragma unroll
            for (int j = 0; j < 4; ++j) wgrad_keep(keep[u >> 2], words[j], limit);
        }
    }
    asm volatile("" : "+v"(keep[0]), "+v"(keep[1]));   // here, not after the products, with the weight spilled until then

    // multiplying: 64 x 64 of a wavefront, 2 x 2 blocks of 32
    const int wk = (wave & 1) * 64, wn = (wave >> 1) * 64, half = lane >> 5;
    int a_at[2], b_at[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int token = half * 8 + ((lane & 15) >> 2), col = i * 32 + ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
        a_at[i] = wgrad_row_slot(token, (wk + col) >> 3) + (col & 4) * 2;
        b_at[i] = kTile + wgrad_row_slot(token, (wn + col) >> 3) + (col & 4) * 2;
    }
    struct Operands { u32x4 a[2], b[2]; };
    auto read = [&](Operands& f, int at, int s) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            u32x2 lo = lds_transposed(lds + at + a_at[i] + s * 4096), hi = lds_transposed(lds + at + a_at[i] + s * 4096 + 1024);
            f.a[i] = u32x4{lo.x, lo.y, hi.x, hi.y};
            lo = lds_transposed(lds + at + b_at[i] + s * 4096);
            hi = lds_transposed(lds + at + b_at[i] + s * 4096 + 1024);
            f.b[i] = u32x4{lo.x, lo.y, hi.x, hi.y};
        }
    };
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    auto multiply = [&](const Operands& f) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = mfma_32x32x16<DT>(f.a[i], f.b[j], acc[i][j]);
    };

    int now = 0, next = kStage, after = 2 * kStage;   // LDS stages: multiplied, complete, being written
    Operands f0, f1;
    // One step: r holds the step after the next, and then the loads of the second one behind that
    auto step = [&](Stage& r) {
        read(f1, now, 1);
        store_x(r, after);
        multiply(f0);
        __builtin_amdgcn_sched_barrier(0);
        read(f0, next, 0);
        store_y(r, after);
        load(r);
        multiply(f1);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        const int free = now;
        now = next;
        next = after;
        after = free;
    };
    store_x(r0, now);
    store_y(r0, now);
    load(r0);
    store_x(r1, next);
    store_y(r1, next);
    load(r1);
    __syncthreads();
    read(f0, now, 0);
    for (int64_t t = 0; t < tokens; t += 2 * kWgLongTokens) {   // tokens past the end are zeros
        step(r0);
        step(r1);
    }
    __syncthreads();   // the operands read ahead of the loop's end

    wgrad_results<DT>(lds, acc, wn, wk, lane);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int row = u * 16 + out_row;
        u32x4 g = wgrad_result(lds, row, out_chunk);
#pragma unroll
        for (int j = 0; j < 4; ++j) g[j] &= wgrad_mask(keep[u >> 2] >> ((u & 3) * 4 + j));
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
#define CALL(KERNEL, DT)                                                                                    \
    mo::KERNEL<DT><<<(unsigned)(tn * tk), 256, 0, s>>>(                                                     \
        (const uint16_t*)dy, (const uint16_t*)x, (const uint16_t*)w, (uint16_t*)dw, tokens, n, k, (uint32_t)tn, \
        (uint32_t)tk, amax, amax_dtype, (uint32_t)inner, narrow_amax)
    // From where it is faster at every size measured (16 shapes, both types, 384 to 4096 tokens: at 384 bf16 14336 x 4096 92.8 -> 82.1 us,
    // 4096 x 64 9.2 -> 8.5, 2752 x 4096 20.7 -> 19.9; at 256 14336 x 4096 62 and 62), and where 32 rows have 32-bit byte offsets
    if (tokens >= 384 && n < 1 << 25 && k < 1 << 25) {
        if (dtype == MO_BF16) CALL(wgrad_masked_long_kernel, MO_BF16); else CALL(wgrad_masked_long_kernel, MO_F16);
    } else {
        if (dtype == MO_BF16) CALL(wgrad_masked_kernel, MO_BF16); else CALL(wgrad_masked_kernel, MO_F16);
    }
#undef CALL
    return hipGetLastError() == hipSuccess ? MO_OK : MO_ERR_LAUNCH;
}
