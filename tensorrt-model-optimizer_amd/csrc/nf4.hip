// NF4 (4-bit table codes, block abs-max scales) quantise+pack and dequantise for gfx950.
// HBM-bound elementwise work; numerics are those of the reference's CPU torch path.
//
// Quantise, per block of `bs` flat elements (zero padded to a whole block):
//   scale = max |x|                                  (stored in the input dtype)
//   v     = T(f32(x) / f32(scale))                   (T = input dtype)
//   code  = first index of the minimum of T(|v - table[i]|), i = 0..15; index 0 when v is NaN
//   byte  = code[2i] << 4 | code[2i + 1]
// The table is the bf16 rounding of the sixteen NF4 constants.  Its entries are at least 0.079
// apart and |v| <= 1, so only the two entries that bracket v can share the minimum, and
// whether the upper one wins is monotone in v: for each pair of neighbours there is one
// threshold t[j] with "upper wins <=> v > t[j]", and code = number of thresholds below v.
// The thresholds depend on T (the differences are rounded to T) and are found on the host by
// bisection on exactly the comparison above; fp32 does a four-step binary search over them.
#include "common.h"

namespace mo {

struct Nf4Thresholds { float t[15]; };

// bf16(-1, -0.6962, -0.5251, -0.3949, -0.2844, -0.1848, -0.0911, 0, 0.0796, 0.1609, 0.2461,
//      0.3379, 0.4407, 0.5626, 0.7230, 1)
#define MO_NF4_TABLE                                                                           \
    {-1.0f, -0.6953125f, -0.5234375f, -0.39453125f, -0.28515625f, -0.1845703125f,              \
     -0.09130859375f, 0.0f, 0.07958984375f, 0.1611328125f, 0.24609375f, 0.337890625f,          \
     0.44140625f, 0.5625f, 0.72265625f, 1.0f}

__device__ __constant__ float kNf4Table[16] = MO_NF4_TABLE;

template <int VIA>
__device__ __forceinline__ float nf4_round_via(float v) {
    if constexpr (VIA == MO_BF16) return bf16_bits_to_f32(f32_to_bf16_bits(v));
    else if constexpr (VIA == MO_F16) return f16_bits_to_f32(f32_to_f16_bits(v));
    else return v;
}

// The thresholds as fifteen register values.  They are handed on as separate scalars, never
// through a pointer or reference: selecting between two of them must stay a select of values
// (given an address the compiler turns it into a load at a selected address, and the copy of
// the argument struct then lives in scratch memory).
struct Nf4Regs {
    float t0, t1, t2, t3, t4, t5, t6, t7, t8, t9, t10, t11, t12, t13, t14;
};

__device__ __forceinline__ Nf4Regs nf4_regs(const Nf4Thresholds& th) {
    float f[15];
#pragma unroll
    for (int j = 0; j < 15; ++j) {
        f[j] = th.t[j];
        asm volatile("" : "+v"(f[j]));
    }
    return {f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7], f[8], f[9], f[10], f[11], f[12],
            f[13], f[14]};
}

// number of thresholds below v (NaN: none)
__device__ __forceinline__ uint32_t nf4_code_scalars(float v, float t0, float t1, float t2,
                                                     float t3, float t4, float t5, float t6,
                                                     float t7, float t8, float t9, float t10,
                                                     float t11, float t12, float t13, float t14) {
    const bool b3 = v > t7;
    const bool b2 = v > (b3 ? t11 : t3);
    const float m1 = b3 ? (b2 ? t13 : t9) : (b2 ? t5 : t1);
    const bool b1 = v > m1;
    const float m0 = b3 ? (b2 ? (b1 ? t14 : t12) : (b1 ? t10 : t8))
                        : (b2 ? (b1 ? t6 : t4) : (b1 ? t2 : t0));
    const bool b0 = v > m0;
    return (b3 ? 8u : 0u) | (b2 ? 4u : 0u) | (b1 ? 2u : 0u) | (b0 ? 1u : 0u);
}

#define nf4_code(v, R)                                                                         \
    nf4_code_scalars(v, (R).t0, (R).t1, (R).t2, (R).t3, (R).t4, (R).t5, (R).t6, (R).t7, (R).t8, \
                     (R).t9, (R).t10, (R).t11, (R).t12, (R).t13, (R).t14)

template <int DT>
__device__ __forceinline__ uint32_t nf4_codes8(const float (&v)[8], float amax, Nf4Regs th) {
    const float r = 1.0f / amax;
    const bool fast = mid_range(amax);  // finite, non-zero, no under- or overflow in the FMAs
    uint32_t w = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float q = fast ? exact_quotient(v[j], amax, r) : v[j] / amax;
        const uint32_t c = nf4_code(nf4_round_via<DT>(q), th);
        w |= c << (4 * (j ^ 1));  // even element of a pair in the high nibble of its byte
    }
    return w;
}

// One lane per block: any even block size, zero padding of the last block.
template <int DT>
__global__ __launch_bounds__(256) void nf4_quantize_kernel(const void* __restrict__ x, int64_t n,
                                                           int64_t bs, int64_t nblocks,
                                                           Nf4Thresholds thresholds,
                                                           void* __restrict__ scales,
                                                           uint8_t* __restrict__ packed) {
    const Nf4Regs th = nf4_regs(thresholds);
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; b < nblocks; b += stride) {
        const int64_t i0 = b * bs;
        uint32_t m = 0;
        for (int64_t j = 0; j < bs; ++j) {
            const float v = i0 + j < n ? load_elem<DT>(x, i0 + j) : 0.0f;
            const uint32_t t = f2u(v) & 0x7FFFFFFFu;
            m = t > m ? t : m;
        }
        const float amax = u2f(m);
        store_elem<DT>(scales, b, amax);
        for (int64_t j = 0; j < bs; j += 2) {
            uint32_t c[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float v = i0 + j + h < n ? load_elem<DT>(x, i0 + j + h) : 0.0f;
                c[h] = nf4_code(nf4_round_via<DT>(v / amax), th);
            }
            packed[(i0 + j) >> 1] = (uint8_t)((c[0] << 4) | c[1]);
        }
    }
}

// Tile form: block size 8 << shift with no padding; a lane owns chunks of 8 elements, the
// lanes of a block share their maximum through DPP moves, loads are issued before any math.
constexpr int kNf4TileChunks = 1024;

template <int DT>
__global__ __launch_bounds__(256) void nf4_quantize_tile_kernel(
    const void* __restrict__ x, int64_t chunks, int lanes_per_block, int shift,
    Nf4Thresholds thresholds, void* __restrict__ scales, uint32_t* __restrict__ packed) {
    const Nf4Regs th = nf4_regs(thresholds);
    const int64_t c0 = (int64_t)blockIdx.x * kNf4TileChunks + threadIdx.x;
    RawChunk<DT> raw[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int64_t c = c0 + u * 256;
        zero_raw<DT>(raw[u]);
        if (c < chunks) load_raw<DT>(x, c << 3, raw[u]);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int64_t c = c0 + u * 256;
        float v[8];
        unpack_raw<DT>(raw[u], v);
        uint32_t m = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t t = f2u(v[j]) & 0x7FFFFFFFu;
            m = t > m ? t : m;
        }
        // chunks is a multiple of lanes_per_block, so the lanes of a block are all in or all out
        m = group_max_u32(m, shift);
        if (c >= chunks) continue;
        const float amax = u2f(m);
        if ((threadIdx.x & (lanes_per_block - 1)) == 0) store_elem<DT>(scales, c >> shift, amax);
        __builtin_nontemporal_store(nf4_codes8<DT>(v, amax, th), packed + c);
    }
}

// The 16-bit dtypes.  The code of x under block abs-max a is the number of boundaries m[j] below x / a
// (at m[j] itself where the tie rounds to the upper side), m[j] the point between two neighbours of
// type T where the comparison above tips: 9 significant bits (bf16) or 12 (fp16).  m[j] * a then fits
// fp32 exactly, so the side of x is the sign of x - m[j] * a, one FMA without an error in its sign;
// and x / a is either m[j] or at least 2^-23 of it away, so the rounding of the quotient to fp32 never
// crosses a boundary.  Which boundary to ask follows from x / a to within 1/32: a bucket of 1/16 holds one
// boundary at most (they are 0.08 apart), and an approximate quotient is enough since neighbouring buckets
// both hold a boundary near their common edge.  Seven vector instructions and one conflict-free LDS
// read of 8 bytes an element.  14336 x 4096 bf16: 25.7 us (5.7 TB/s); with the code
// of every 16-bit quotient in a 32 KB LDS table, an exact quotient and its rounding an element, 40.7 us.
constexpr int kNf4Buckets = 33;   // round(16 * x / a) + 16
struct Nf4Bucket { float m; uint32_t edge; };
struct Nf4Buckets { Nf4Bucket b[kNf4Buckets]; };

template <int DT>
__device__ __forceinline__ uint32_t chunk_max_bits(const RawChunk<DT>& r) {
    uint32_t t = pk_max_u16(pk_max_u16(r.a.x & 0x7FFF7FFFu, r.a.y & 0x7FFF7FFFu),
                            pk_max_u16(r.a.z & 0x7FFF7FFFu, r.a.w & 0x7FFF7FFFu));
    t = (t & 0xFFFFu) > (t >> 16) ? (t & 0xFFFFu) : (t >> 16);
    return DT == MO_BF16 ? t << 16 : f2u(f16_bits_to_f32(t));
}

template <int DT>
__global__ __launch_bounds__(256) void nf4_quantize_buckets_kernel(
    const void* __restrict__ x, int64_t chunks, int lanes_per_block, int shift, Nf4Thresholds thresholds,
    Nf4Buckets buckets, void* __restrict__ scales, uint32_t* __restrict__ packed) {
    __shared__ Nf4Bucket tab[kNf4Buckets];
    const int64_t c0 = (int64_t)blockIdx.x * kNf4TileChunks + threadIdx.x;
    RawChunk<DT> raw[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int64_t c = c0 + u * 256;
        zero_raw<DT>(raw[u]);
        if (c < chunks) load_raw<DT>(x, c << 3, raw[u]);
    }
    if (threadIdx.x < kNf4Buckets) tab[threadIdx.x] = buckets.b[threadIdx.x];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int64_t c = c0 + u * 256;
        float v[8];
        unpack_raw<DT>(raw[u], v);
        // chunks is a multiple of lanes_per_block, so the lanes of a block are all in or all out
        const float amax = u2f(group_max_u32(chunk_max_bits<DT>(raw[u]), shift));
        if (c >= chunks) continue;
        if ((threadIdx.x & (lanes_per_block - 1)) == 0) store_elem<DT>(scales, c >> shift, amax);
        uint32_t w = 0;
        if (mid_range(amax)) {
            const float r16 = 16.0f / amax;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int j = i ^ 1;   // even element of a pair in the high nibble of its byte
                // the rounding of the sum leaves the bucket number in the low mantissa bits
                const uint32_t k = f2u(__builtin_fmaf(v[j], r16, 12582912.0f + 16.0f)) - 0x4B400000u;
                const Nf4Bucket e = tab[k];
                const float d = __builtin_fmaf(-e.m, amax, v[j]);
                // the sign of the tiny edge says which side d == 0 is on, its low bits are the code below
                const uint32_t code = e.edge + (d > u2f(e.edge) ? 1u : 0u);
                w = __builtin_amdgcn_alignbit(code, w, 4);
            }
        } else {
            keep_branch();
            w = nf4_codes8<DT>(v, amax, nf4_regs(thresholds));   // zero, tiny or not finite
        }
        __builtin_nontemporal_store(w, packed + c);
    }
}

// Double-quantised scales, one wavefront per scale block: everything behind the mean, with every
// intermediate rounded to the type of the scales as the tensor expression rounds it
// (T(s - mean), abs-max, T(T(1 / amax) * bound), T(product), round, clamp).  Nine launches of a
// few microseconds each as tensor operations (37 us with their gaps for 3584 x 256 bf16), 5.2 us here.
template <int DT>
__global__ __launch_bounds__(256) void nf4_scales_quantize_kernel(const void* __restrict__ scales, int64_t rows,
                                                                  int width, const void* __restrict__ mean,
                                                                  float bound, int8_t* __restrict__ q,
                                                                  void* __restrict__ factor) {
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int lane = threadIdx.x & 63;
    const float z = load_elem<DT>(mean, 0);
    const int64_t base = row * width;
    uint32_t m = 0;
    for (int i = lane; i < width; i += 64) {
        const uint32_t t = f2u(nf4_round_via<DT>(load_elem<DT>(scales, base + i) - z)) & 0x7FFFFFFFu;
        m = t > m ? t : m;
    }
    for (int o = 32; o > 0; o >>= 1) {
        const uint32_t t = __shfl_xor(m, o, 64);
        m = t > m ? t : m;
    }
    const float f = nf4_round_via<DT>(nf4_round_via<DT>(1.0f / u2f(m)) * bound);
    if (lane == 0) store_elem<DT>(factor, row, f);
    for (int i = lane; i < width; i += 64) {
        const float b = nf4_round_via<DT>(load_elem<DT>(scales, base + i) - z);
        float v = __builtin_rintf(nf4_round_via<DT>(b * f));
        v = v < -bound ? -bound : (v > bound ? bound : v);
        q[base + i] = v == v ? (int8_t)(int)v : (int8_t)0;
    }
}

// T(T(q / factor) + mean): the scale of a block from its int8 form
template <int DT>
__device__ __forceinline__ float nf4_scale_of(int8_t q, float factor, float mean) {
    return nf4_round_via<DT>(nf4_round_via<DT>((float)q / factor) + mean);
}

// y[2i] = T(table[byte >> 4] * f32(scale[block])), y[2i + 1] = T(table[byte & 15] * ...)
template <int DT>
__global__ __launch_bounds__(256) void nf4_dequantize_kernel(const uint8_t* __restrict__ packed,
                                                             int64_t nbytes, int64_t bs,
                                                             const void* __restrict__ scales,
                                                             void* __restrict__ y) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nbytes; i += stride) {
        const uint32_t b = packed[i];
        const float s = load_elem<DT>(scales, (2 * i) / bs);
        store_elem<DT>(y, 2 * i, kNf4Table[b >> 4] * s);
        store_elem<DT>(y, 2 * i + 1, kNf4Table[b & 0xFu] * s);
    }
}

// DOUBLE: int8 scales, decoded on the way (one division per 8 elements): `width` of them share a factor.
// 14336 x 4096 bf16 in blocks of 64: 29.6 us, 28.2 with decoded scales; decoding them first was a division
// and a sum as tensor operations, 12 us and two launches.
template <int DT, bool DOUBLE>
__global__ __launch_bounds__(256) void nf4_dequantize_tile_kernel(
    const uint32_t* __restrict__ packed, int64_t chunks, int shift,
    const void* __restrict__ scales, uint32_t width, const void* __restrict__ factor,
    const void* __restrict__ mean, void* __restrict__ y) {
    __shared__ float table[16];
    if (threadIdx.x < 16) table[threadIdx.x] = kNf4Table[threadIdx.x];
    __syncthreads();
    const int64_t c0 = (int64_t)blockIdx.x * kNf4TileChunks + threadIdx.x;
    uint32_t w[4];
    float sc[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        int64_t c = c0 + u * 256;
        c = c < chunks ? c : chunks - 1;
        w[u] = __builtin_nontemporal_load(packed + c);
        const int64_t b = c >> shift;
        if constexpr (DOUBLE)
            sc[u] = nf4_scale_of<DT>(((const int8_t*)scales)[b], load_elem<DT>(factor, (uint32_t)b / width),
                                     load_elem<DT>(mean, 0));
        else
            sc[u] = load_elem<DT>(scales, b);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int64_t c = c0 + u * 256;
        if (c >= chunks) continue;
        const float s = sc[u];
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = table[(w[u] >> (4 * (j ^ 1))) & 0xFu] * s;
        store_chunk<DT>(y, c << 3, v);
    }
}

// ------------------------------------------------------------------------------ host side
static float host_round(float f, int dtype) {
    if (dtype == MO_F32 || f != f) return f;
    uint32_t u;
    __builtin_memcpy(&u, &f, 4);
    if (dtype == MO_BF16) {
        u += 0x7FFFu + ((u >> 16) & 1u);
        u &= 0xFFFF0000u;
    } else {
        const float a = __builtin_fabsf(f);
        if (a < 6.103515625e-05f) {  // fp16 subnormal range: multiples of 2^-24
            return __builtin_rintf(f * 16777216.0f) * 5.9604644775390625e-08f;
        }
        u += 0xFFFu + ((u >> 13) & 1u);
        u &= 0xFFFFE000u;
        float g;
        __builtin_memcpy(&g, &u, 4);
        if (__builtin_fabsf(g) > 65504.0f) return f < 0 ? -__builtin_inff() : __builtin_inff();
        return g;
    }
    __builtin_memcpy(&f, &u, 4);
    return f;
}

// fp32 values in numeric order <-> integers in the same order
static int64_t ordered_key(float f) {
    uint32_t u;
    __builtin_memcpy(&u, &f, 4);
    return (u & 0x80000000u) ? -(int64_t)(u & 0x7FFFFFFFu) : (int64_t)u;
}

static float from_key(int64_t k) {
    const uint32_t u = k < 0 ? (0x80000000u | (uint32_t)(-k)) : (uint32_t)k;
    float f;
    __builtin_memcpy(&f, &u, 4);
    return f;
}

// t[j] = the largest fp32 p for which table[j] still wins against table[j + 1] at v = T(p)
static Nf4Thresholds nf4_thresholds(int dtype) {
    static const float table[16] = MO_NF4_TABLE;
    Nf4Thresholds th;
    for (int j = 0; j < 15; ++j) {
        auto upper_wins = [&](float p) {
            const float v = host_round(p, dtype);
            const float lo = host_round(__builtin_fabsf(v - table[j]), dtype);
            const float hi = host_round(__builtin_fabsf(v - table[j + 1]), dtype);
            return hi < lo;
        };
        int64_t a = ordered_key(table[j]), b = ordered_key(table[j + 1]);  // false at a, true at b
        while (b - a > 1) {
            const int64_t mid = a + (b - a) / 2;
            if (upper_wins(from_key(mid))) b = mid; else a = mid;
        }
        th.t[j] = from_key(a);
    }
    return th;
}

// The buckets of a 16-bit type from its thresholds.  t[j] is the largest fp32 value on the lower side: the
// boundary itself when that side has the tie, the value just below it otherwise.
static Nf4Buckets nf4_buckets(int dtype, const Nf4Thresholds& th) {
    const uint32_t rest = dtype == MO_BF16 ? 0x7FFFu : 0xFFFu;   // mantissa bits below a boundary's last one
    float m[15];
    bool upper_has_tie[15];
    for (int j = 0; j < 15; ++j) {
        uint32_t u;
        __builtin_memcpy(&u, &th.t[j], 4);
        upper_has_tie[j] = (u & rest) != 0;
        m[j] = upper_has_tie[j] ? from_key(ordered_key(th.t[j]) + 1) : th.t[j];
    }
    Nf4Buckets out;
    for (int i = 0; i < kNf4Buckets; ++i) {
        const double lo = (i - 16.5) / 16.0 - 1e-4, hi = (i - 15.5) / 16.0 + 1e-4;
        uint32_t below = 0;
        while (below < 15 && m[below] < lo) ++below;
        const bool inside = below < 15 && m[below] <= hi;
        out.b[i].m = inside ? m[below] : 2.0f;   // x - 2 * amax is negative: the code below it stands
        // +-2^-120: far below any difference of two values of the type within the range of the buckets
        out.b[i].edge = (inside && upper_has_tie[below] ? 0x83800000u : 0x03800000u) | below;
    }
    return out;
}

struct Nf4Tables {
    Nf4Thresholds th;
    Nf4Buckets buckets;
};

// built once per type: a function-local constant, initialised under the language's own lock
static const Nf4Tables& nf4_tables(int dtype) {
    static const auto make = [](int d) {
        Nf4Tables t;
        t.th = nf4_thresholds(d);
        t.buckets = d == MO_F32 ? Nf4Buckets{} : nf4_buckets(d, t.th);
        return t;
    };
    static const Nf4Tables tables[3] = {make(MO_F32), make(MO_F16), make(MO_BF16)};
    return tables[dtype];
}

static inline unsigned nf4_blocks_for(int64_t items) {
    int64_t b = (items + 255) / 256;
    if (b < 1) b = 1;
    if (b > 65536) b = 65536;
    return (unsigned)b;
}

}  // namespace mo

#define DISPATCH_DT(dtype, CALL)        \
    switch (dtype) {                    \
        case MO_F32: CALL(MO_F32); break; \
        case MO_F16: CALL(MO_F16); break; \
        case MO_BF16: CALL(MO_BF16); break; \
        default: return MO_ERR_DTYPE;   \
    }

extern "C" int mo_nf4_quantize(const void* x, int64_t n, int64_t block_size, int dtype,
                               void* scales, uint8_t* packed, void* stream) {
    if (n < 0 || block_size <= 0 || (block_size & 1)) return MO_ERR_ARG;
    if (dtype != MO_F32 && dtype != MO_F16 && dtype != MO_BF16) return MO_ERR_DTYPE;
    if (n == 0) return MO_OK;
    if (!x || !scales || !packed) return MO_ERR_ARG;
    const int64_t nblocks = (n + block_size - 1) / block_size;
    hipStream_t s = (hipStream_t)stream;
    const mo::Nf4Tables& tables = mo::nf4_tables(dtype);
    const mo::Nf4Thresholds& th = tables.th;
    int shift = -1;  // block_size == 8 << shift
    for (int k = 0; k <= 6; ++k)
        if (block_size == (8ll << k)) shift = k;
    const int64_t tiles = (n / 8 + mo::kNf4TileChunks - 1) / mo::kNf4TileChunks;
    if (shift >= 0 && n % block_size == 0 && (((uintptr_t)x & 15u) == 0) &&
        (((uintptr_t)packed & 3u) == 0) && tiles <= 0x7FFFFFFF) {
#define CALL(DT)                                                                    \
    mo::nf4_quantize_buckets_kernel<DT><<<(unsigned)tiles, 256, 0, s>>>(            \
        x, n / 8, 1 << shift, shift, th, tables.buckets, scales, (uint32_t*)packed)
        if (dtype == MO_BF16) CALL(MO_BF16);
        else if (dtype == MO_F16) CALL(MO_F16);
        else
            mo::nf4_quantize_tile_kernel<MO_F32><<<(unsigned)tiles, 256, 0, s>>>(
                x, n / 8, 1 << shift, shift, th, scales, (uint32_t*)packed);
#undef CALL
        return hipGetLastError() == hipSuccess ? MO_OK : MO_ERR_LAUNCH;
    }
    const unsigned g = mo::nf4_blocks_for(nblocks);
#define CALL(DT) mo::nf4_quantize_kernel<DT><<<g, 256, 0, s>>>(x, n, block_size, nblocks, th, scales, packed)
    DISPATCH_DT(dtype, CALL)
#undef CALL
    return hipGetLastError() == hipSuccess ? MO_OK : MO_ERR_LAUNCH;
}

extern "C" int mo_nf4_scales_quantize(const void* scales, int64_t rows, int64_t width, int dtype,
                                      const void* mean, int bound, int8_t* q, void* factor, void* stream) {
    if (rows < 0 || width < 0 || bound < 1 || bound > 127) return MO_ERR_ARG;
    if (dtype != MO_F32 && dtype != MO_F16 && dtype != MO_BF16) return MO_ERR_DTYPE;
    if (rows == 0 || width == 0) return MO_OK;
    if (!scales || !mean || !q || !factor) return MO_ERR_ARG;
    if (width > 0x3FFFFFFF || rows > 0x7FFFFFFFll * 4) return MO_ERR_UNSUPPORTED;
    const unsigned g = (unsigned)((rows + 3) / 4);
#define CALL(DT)                                                                    \
    mo::nf4_scales_quantize_kernel<DT><<<g, 256, 0, (hipStream_t)stream>>>(         \
        scales, rows, (int)width, mean, (float)bound, q, factor)
    DISPATCH_DT(dtype, CALL)
#undef CALL
    return hipGetLastError() == hipSuccess ? MO_OK : MO_ERR_LAUNCH;
}

static int nf4_dequantize(const uint8_t* packed, int64_t nbytes, int64_t block_size, const void* scales,
                          int64_t width, const void* factor, const void* mean, void* y, int dtype, void* stream) {
    if (nbytes < 0 || block_size <= 0 || (block_size & 1)) return MO_ERR_ARG;
    if (dtype != MO_F32 && dtype != MO_F16 && dtype != MO_BF16) return MO_ERR_DTYPE;
    if (nbytes == 0) return MO_OK;
    if (!packed || !scales || !y) return MO_ERR_ARG;
    hipStream_t s = (hipStream_t)stream;
    int shift = -1;
    for (int k = 0; k <= 40; ++k)
        if (block_size == (8ll << k)) shift = k;
    const int64_t tiles = (nbytes / 4 + mo::kNf4TileChunks - 1) / mo::kNf4TileChunks;
    if (shift >= 0 && nbytes % 4 == 0 && (((uintptr_t)y & 15u) == 0) &&
        (((uintptr_t)packed & 3u) == 0) && tiles <= 0x7FFFFFFF) {
        if (factor && ((nbytes / 4) >> shift) > 0xFFFFFFFFll) return MO_ERR_UNSUPPORTED;
#define CALL(DT)                                                                           \
    if (factor)                                                                            \
        mo::nf4_dequantize_tile_kernel<DT, true><<<(unsigned)tiles, 256, 0, s>>>(          \
            (const uint32_t*)packed, nbytes / 4, shift, scales, (uint32_t)width, factor, mean, y); \
    else                                                                                   \
        mo::nf4_dequantize_tile_kernel<DT, false><<<(unsigned)tiles, 256, 0, s>>>(         \
            (const uint32_t*)packed, nbytes / 4, shift, scales, 1u, nullptr, nullptr, y)
        DISPATCH_DT(dtype, CALL)
#undef CALL
        return hipGetLastError() == hipSuccess ? MO_OK : MO_ERR_LAUNCH;
    }
    if (factor) return MO_ERR_UNSUPPORTED;
    const unsigned g = mo::nf4_blocks_for(nbytes);
#define CALL(DT) mo::nf4_dequantize_kernel<DT><<<g, 256, 0, s>>>(packed, nbytes, block_size, scales, y)
    DISPATCH_DT(dtype, CALL)
#undef CALL
    return hipGetLastError() == hipSuccess ? MO_OK : MO_ERR_LAUNCH;
}

extern "C" int mo_nf4_dequantize(const uint8_t* packed, int64_t nbytes, int64_t block_size,
                                 const void* scales, void* y, int dtype, void* stream) {
    return nf4_dequantize(packed, nbytes, block_size, scales, 1, nullptr, nullptr, y, dtype, stream);
}

extern "C" int mo_nf4_dequantize_double(const uint8_t* packed, int64_t nbytes, int64_t block_size,
                                        const int8_t* scales, int64_t width, const void* factor,
                                        const void* mean, void* y, int dtype, void* stream) {
    if (width < 1 || width > 0x7FFFFFFF || (nbytes > 0 && (!factor || !mean))) return MO_ERR_ARG;
    return nf4_dequantize(packed, nbytes, block_size, scales, width, factor, mean, y, dtype, stream);
}
