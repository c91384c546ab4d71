// AWQ clip search for gfx950: for every weight block and every clip ratio, the squared error the
// clipped, fake-quantised block makes on the block's partial outputs over the calibration
// tokens -- one launch per batch of tokens instead of (ratios x row batches) broadcast products.
//
// What is computed, in the dtype T of the weight (all as the tensor expression would round):
//   org[t]  = T( sum_j T(x[t, j] * w[j]) )                 j over the block, fp32 accumulation
//   cur[t]  = T( sum_j T(x[t, j] * wq_r[j]) )              wq_r = T(qdq(w; T(f32(amax) * r)))
//   loss[r] += ( sum_t f32(T(cur[t] - org[t]))^2 ) / tokens
//
// Every product is rounded to T before it is summed, so the products themselves cannot be one
// contraction; what the matrix cores can do is make the products (an outer product per column j,
// whose fp32 result is exact for 16-bit operands) and add them up once they are rounded (a
// contraction with a 0 / 1 matrix).  Issue costs, measured per wavefront instruction: 4.5 cycles for
// v_mul_f32, v_cvt_pk_bf16_f32, v_pk_mul_f16 and v_dot2c, 16 cycles for a 16x16x32, 32 for a
// 32x32x16 and 64 for a 32x32x4 (two blocks) matrix instruction, which run beside the vector instructions of
// other wavefronts and take about 8 cycles of the issue port themselves.
//   bf16: products on the matrix cores, one conversion per two products on the vector ALU, sums on the
//         matrix cores (clip_losses_bf16): 0.5 vector instructions per product where multiply,
//         convert and v_dot2c took 2.
//   fp16: v_pk_mul_f16 rounds two products at once, sums on the matrix cores (clip_losses_f16): 0.5
//         vector instructions per product where multiply, round and add took about 4.
//   fp32: no rounding to do, one multiply and one add per product (clip_losses_f32).
// A sum by selection leaves most of a matrix instruction idle: a dense one takes 512 products and adds two of them to
// each of 256 sums.  The sparse form (v_smfmac, two of every four k) takes 1024 in the same 16 cycles: the
// operand that says which is the sparse one, the products are the dense one.  It adds the two pairs of a sum one
// after the other and leaves the bits of two dense instructions.
// Measured, 4096 x 4096, 64 tokens, 11 ratios, dense / sparse: bf16 blocks of 128 495 / 400 - 414 us, of 64 520 / 425, of 16
// 620 / 517; fp16 442 / 440, 436 / 418, 608 / 605.  bf16 blocks of 32 keep the dense form: their chains are so short
// that the words held for the second step and the fold of the chains do not fit the registers of three wavefronts
// a SIMD (50 spill: 1500 us against 537).
// The instruction adds a pair of products to an output with one rounding, as v_dot2c does.  Its sums are made
// in chains of a quarter of a block (but for blocks of 16), as four chains of v_dot2c made them: one
// chain through a block of 128 rounds at twice the magnitude, and measured against sums in 64 bits 41 % more
// blocks had an output that fell on the other side of a rounding to bf16 (1199 of 1.57 million; 852 with
// quarters, 856 with v_dot2c).
// Measured figures stand at the launch below.
#include "common.h"
#include "qdq_ops.h"

namespace mo {

constexpr int kClipMaxRatios = 32;
constexpr int kClipTokens = 64;   // tokens of a pass over the ratios (fp32: per wavefront)
constexpr int kClipLanes = 64;
constexpr int kClipWaves = 4;     // wavefronts of a workgroup (fp32: at most)

struct ClipRatios {
    float r[kClipMaxRatios];
    int count;
};

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x16_t __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x16_t __attribute__((ext_vector_type(16)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x32_t __attribute__((ext_vector_type(32)));

template <int DT>
__device__ __forceinline__ float clip_round(float v) {
    if constexpr (DT == MO_BF16) return round_to_bf16(v);
    else if constexpr (DT == MO_F16) return f16_bits_to_f32(f32_to_f16_bits(v));
    else return v;
}

// The quantiser of one block at one ratio: `w_amax * ratio` on a tensor is an fp32 product rounded
// to the dtype of the amax.
__device__ __forceinline__ IntOp::Scale clip_scale(const IntOp& op, float amax, int amax_dtype, float ratio) {
    float clipped = amax * ratio;
    if (amax_dtype == MO_BF16) clipped = clip_round<MO_BF16>(clipped);
    else if (amax_dtype == MO_F16) clipped = clip_round<MO_F16>(clipped);
    return op.make(clipped);
}

// op.apply where clip_fast says so, less the sign of a zero (the value is only summed)
__device__ __forceinline__ bool clip_fast(const IntOp& op, const IntOp::Scale& s) {
    return s.fast && op.bound <= 2047.0f;   // codes of at most 11 bits: the short quotient
}
__device__ __forceinline__ float clip_qdq_fast(const IntOp& op, float v, const IntOp::Scale& s) {
    const float q = __builtin_amdgcn_fmed3f(__builtin_rintf(v * s.mul), op.lo, op.bound);
    return exact_quotient_short(q, s.div, s.rdiv);
}

// A selection by zeros does not select among products that are not finite: inf * 0 is NaN in every sum of
// its matrix row, the sums of other weight rows among them.  Any such sum ends the quick form of a
// wavefront before the losses of that step are written, and the careful form goes on from there: over
// the products of a step twice, once for their kinds and once without those that are not finite, so that
// the rows without any get the bits they would have alone.  A kind is a power of two whose sums over a block
// (128 at most of each) stay apart in 24 bits; two words of 16 bits at a time, E the exponent mask of the type.
// The forms come one after the other, not one within the other, which would cost the quick one registers.
struct ClipStep {
    int token, ratio;   // first token of the pass, index of the ratio (that of the unclipped block: before the first)
};

template <uint32_t E, uint32_t POS, uint32_t NEG, uint32_t NAN_>
__device__ __forceinline__ uint32_t clip_kinds(uint32_t w, bool kinds) {
    uint32_t out = 0;
#pragma unroll
    for (int h = 0; h < 32; h += 16) {
        const uint32_t v = (w >> h) & 0xFFFFu;
        const bool finite = (v & E) != E;
        const uint32_t kind = (v & 0x7FFFu) != E ? NAN_ : (v & 0x8000u) ? NEG : POS;
        out |= (kinds ? (finite ? 0u : kind) : (finite ? v : 0u)) << h;
    }
    return out;
}
// 2^-8 for +inf, 1 for -inf, 2^8 for NaN
__device__ __forceinline__ uint32_t clip_kinds_bf16(uint32_t w, bool kinds) {
    return clip_kinds<0x7F80u, 0x3B80u, 0x3F80u, 0x4380u>(w, kinds);
}
__device__ __forceinline__ uint32_t clip_kinds_f16(uint32_t w, bool kinds) {
    return clip_kinds<0x7C00u, 0x1C00u, 0x3C00u, 0x5C00u>(w, kinds);
}
// The sum of the products without those, given the kinds among them: 0 none, 1 +inf, 2 -inf, 3 NaN or both
__device__ __forceinline__ uint32_t clip_sum_kind(float kinds) {
    const uint32_t c = (uint32_t)(kinds * 256.0f);
    const uint32_t k = ((c & 0xFFu) ? 1u : 0u) | ((c & 0xFF00u) ? 2u : 0u);
    return c >> 16 ? 3u : k;
}
__device__ __forceinline__ float clip_with_kind(float sum, uint32_t kind) {
    const uint32_t special = kind == 3 ? 0x7FC00000u : 0x7F800000u | (kind & 2u) << 30;
    return kind ? u2f(special) : sum;
}

// The 0 / 1 operand A of a sum, constant through a kernel.  As B the instruction takes eight words of a lane, four sums
// with two words each: word i and word 4 + i.  Row 4 g + i of A picks them out of lane group g (16 lanes), so that
// lane l, register i of the result is the sum of the words of lane l: no value changes its lane.
// Dense (16x16x32): the first four words only.
__device__ __forceinline__ void clip_sum_operand(uint32_t one, uint32_t (&m)[4]) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < 4; ++i) m[i] = (lane & 15) == 4 * (lane >> 4) + i ? one : 0u;
}
// Sparse (16x16x64, two of every four k): B has the first words of lane group g at k = 8 g .. 8 g + 7, the second ones 32
// behind; lane (h, row) of A holds k = 16 h .. 16 h + 15 as four pairs, each pair with the same two places among its four.
__device__ __forceinline__ int clip_sum_operand_sparse(uint32_t one, uint32_t (&m)[4]) {
    const int lane = threadIdx.x & 63, h = lane >> 4, g = (lane >> 2) & 3, i = lane & 3;
#pragma unroll
    for (int p = 0; p < 4; ++p) m[p] = (h & 1) == (g >> 1) && p == (g & 1) * 2 + (i >> 1) ? one : 0u;
    return (i & 1) ? 0xEEEE : 0x4444;   // places 2 and 3, or 0 and 1
}

// ------------------------------------------------------------------------------------- bf16
// A wavefront owns 32 rows of one weight block and all tokens of a pass, in two tiles of 32.  For two
// columns (j, j + 8) of the block, v_mfma_f32_32x32x4_2b_bf16 with the tokens as A, reduced to one of
// its four k by zeroing the others, and the weights as B gives the exact products of 32 tokens x 32
// rows in 32 registers: register i of the first half and of the second half are the same token and
// row under j and j + 8.  One conversion rounds the two into a word.  The words of two steps are the B
// operand of v_smfmac_f32_16x16x64_bf16 (those of one of v_mfma_f32_16x16x32_bf16), four tokens at a time, and
// their lo + hi go to a sum of their own in the same lane: lane l, register i of group a holds
//   row l & 31, token 8 a + 4 (l >> 5) + i
// of the tile.  The sums of the chains that have ended and the partial outputs of the unclipped block lie in
// LDS, each lane's own: no barrier anywhere.  Folding stands where the products before it are used up, or
// its operands would not fit the registers.  The weights are quantised as they are used, 16 columns at a
// time, by the lane that supplies them to the matrix instruction.
template <int BS, bool CAREFUL>
__device__ __forceinline__ bool clip_losses_bf16(const uint16_t* __restrict__ x, int tokens,
                                                 const uint16_t* __restrict__ w, int n, int k,
                                                 const void* __restrict__ w_amax, int amax_dtype,
                                                 const ClipRatios& ratios, int r0, int r1,
                                                 const IntOp& op, float* __restrict__ loss,
                                                 f32x4* __restrict__ parts, u32x2* __restrict__ org, ClipStep& at) {
    constexpr int NC = BS / 16;
    constexpr int HALVES = BS >= 32 ? BS / 32 : 2;   // of a chunk, in a chain of sums
    constexpr bool SPARSE = !CAREFUL && BS != 32;
    constexpr int RUN = HALVES >= 2 ? HALVES / 2 : 1;   // chunks until the chains of both tiles have ended
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int fr = lane & 31;
    const int nblk = k / BS, b = blockIdx.y;
    const int row0 = (blockIdx.x * kClipWaves + wave) * 32;
    if (row0 >= n) return true;
    int row = row0 + fr < n ? row0 + fr : n - 1;
    const float amax = load_scalar(w_amax, amax_dtype, (int64_t)row * nblk + b);
    bf16x8_t picks;
    int places = 0;
    {
        uint32_t m[4];
        if constexpr (!SPARSE) clip_sum_operand(0x3F803F80u, m);
        else places = clip_sum_operand_sparse(0x3F803F80u, m);
        __builtin_memcpy(&picks, m, 16);
    }
    f32x32_t zero;
#pragma unroll
    for (int i = 0; i < 32; ++i) zero[i] = 0.0f;
    for (int t0 = CAREFUL ? __builtin_amdgcn_readfirstlane(at.token) : 0; t0 < tokens; t0 += kClipTokens) {
        bool live[2];   // a token past the end counts as a row of zeros
#pragma unroll
        for (int m = 0; m < 2; ++m) live[m] = t0 + 32 * m + fr < tokens;
        // The addresses are made anew for every chunk from the lane's number: what is kept across the
        // chunk loop beside the sums and the products would cost the third wavefront of a SIMD.
        u32x4 wraw, xraw[2];
        auto fetch = [&](int c) {
            int l = lane;
            asm volatile("" : "+v"(l), "+v"(row));
            const int col = b * BS + c * 16 + (l >> 5) * 8;
            wraw = *(const u32x4*)(w + ((int64_t)row * k + col));
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const int t = t0 + 32 * m + (l & 31);
                xraw[m] = *(const u32x4*)(x + ((int64_t)(t < tokens ? t : tokens - 1) * k + col));
            }
        };
        fetch(0);
        for (int v = r0 - 1; v < r1; ++v) {   // r0 - 1: the unclipped block
            if (CAREFUL && v >= r0 && t0 == at.token && v < at.ratio) continue;   // in the losses already
            IntOp::Scale s = {};
            if (v >= r0) s = clip_scale(op, amax, amax_dtype, ratios.r[v]);
            f32x4 acc[2][4];
            auto clear = [&]() {
#pragma unroll
                for (int m = 0; m < 2; ++m)
#pragma unroll
                    for (int a = 0; a < 4; ++a) parts[(4 * m + a) * 64] = acc[m][a] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            };
            // the end of the chains: their sums go to those of the chains before them
            auto fold = [&]() {
                if (HALVES == 2 * NC) return;
#pragma unroll
                for (int m = 0; m < 2; ++m)
#pragma unroll
                    for (int a = 0; a < 4; ++a) {
                        acc[m][a] = parts[(4 * m + a) * 64] + acc[m][a];
                        parts[(4 * m + a) * 64] = acc[m][a];
                    }
            };
            // the operands of the chunk that was fetched: the weights quantised, the tokens that exist
            auto operands = [&](uint32_t (&wb)[4], uint32_t (&xb)[2][4]) {
                wb[0] = wraw.x, wb[1] = wraw.y, wb[2] = wraw.z, wb[3] = wraw.w;
                if (v >= r0) {
                    float q[8];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        q[2 * j] = u2f(wb[j] << 16);
                        q[2 * j + 1] = u2f(wb[j] & 0xFFFF0000u);
                    }
                    // the choice between the exact-reciprocal quotient and a division is per block
                    if (clip_fast(op, s)) {
#pragma unroll
                        for (int j = 0; j < 8; ++j) q[j] = clip_qdq_fast(op, q[j], s);
                    } else {
                        keep_branch();
#pragma unroll
                        for (int j = 0; j < 8; ++j) q[j] = op.apply<false>(q[j], s);
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) wb[j] = f32x2_to_bf16x2(q[2 * j], q[2 * j + 1]);
                }
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    xb[m][0] = live[m] ? xraw[m].x : 0u;
                    xb[m][1] = live[m] ? xraw[m].y : 0u;
                    xb[m][2] = live[m] ? xraw[m].z : 0u;
                    xb[m][3] = live[m] ? xraw[m].w : 0u;
                }
            };
            // Step q of a chunk: four columns of its lower half and the same of its upper half, of either
            // tile of tokens in turn, then the other four
            auto products = [&](const uint32_t (&wb)[4], const uint32_t (&xb)[2][4], int q) {
                const int m = (q >> 2) & 1, e = (q >> 3) * 4 + (q & 3);
                const uint32_t one = xb[m][e >> 1] & ((e & 1) ? 0xFFFF0000u : 0x0000FFFFu);
                const uint32_t aw[2] = {(e & 2) ? 0u : one, (e & 2) ? one : 0u};
                const uint32_t bw[2] = {wb[(e >> 2) * 2], wb[(e >> 2) * 2 + 1]};
                s16x4_t av, bv;
                __builtin_memcpy(&av, aw, 8);
                __builtin_memcpy(&bv, bw, 8);
                return __builtin_amdgcn_mfma_f32_32x32x4bf16_1k(av, bv, zero, 0, 0, 0);
            };
            if constexpr (CAREFUL) {
                uint32_t kind[2] = {0, 0};   // two bits an output
#pragma unroll 1
                for (int pass = 0; pass < 2; ++pass) {
                    clear();
#pragma unroll 1
                    for (int c = 0; c < NC; ++c) {
                        uint32_t wb[4], xb[2][4];
                        fetch(c);
                        operands(wb, xb);
#pragma unroll
                        for (int q = 0; q < 16; ++q) {
                            const int m = (q >> 2) & 1;
                            const bool opens = (c * 2 + (q >> 3)) % HALVES == 0 && (q & 3) == 0;
                            const f32x32_t d = products(wb, xb, q);
#pragma unroll
                            for (int a = 0; a < 4; ++a) {
                                if (opens) acc[m][a] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                                uint32_t pw[4];
#pragma unroll
                                for (int i = 0; i < 4; ++i)
                                    pw[i] = clip_kinds_bf16(f32x2_to_bf16x2(d[4 * a + i], d[16 + 4 * a + i]), pass == 0);
                                bf16x8_t pv;
                                __builtin_memcpy(&pv, pw, 16);
                                acc[m][a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(picks, pv, acc[m][a], 0, 0, 0);
                            }
                            __builtin_amdgcn_sched_barrier(0);
                            if ((c * 2 + (q >> 3)) % HALVES == HALVES - 1 && (q & 7) == 7) fold();
                        }
                    }
#pragma unroll
                    for (int m = 0; m < 2; ++m)
#pragma unroll
                        for (int a = 0; a < 4; ++a)
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                const int bit = 2 * (4 * a + i);
                                if (pass == 0) kind[m] |= clip_sum_kind(acc[m][a][i]) << bit;
                                else acc[m][a][i] = clip_with_kind(acc[m][a][i], (kind[m] >> bit) & 3u);
                            }
                }
            } else {
                clear();
#pragma unroll 1
                for (int c = 0; c < NC; c += RUN) {
#pragma unroll
                    for (int cc = 0; cc < RUN; ++cc) {
                        uint32_t wb[4], xb[2][4];
                        operands(wb, xb);
                        f32x32_t d = products(wb, xb, 0);
                        uint32_t pw[4][8];   // of two steps
#pragma unroll
                        for (int q = 0; q < 16; ++q) {
                            const int m = (q >> 2) & 1, half = cc * 2 + (q >> 3);
                            f32x32_t ahead;   // the next products run under this step's conversions
                            if (q + 1 < 16) ahead = products(wb, xb, q + 1);
                            // half a chunk ahead; the first one again for the next ratio
                            if (q == 8) fetch(c + cc + 1 < NC ? c + cc + 1 : 0);
                            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                            for (int a = 0; a < 4; ++a) {
#pragma unroll
                                for (int i = 0; i < 4; ++i)
                                    pw[a][(SPARSE ? q & 1 : 0) * 4 + i] = f32x2_to_bf16x2(d[4 * a + i], d[16 + 4 * a + i]);
                                if constexpr (!SPARSE) {
                                    const bool opens = half % HALVES == 0 && (q & 3) == 0;
                                    const f32x4 none = {0.0f, 0.0f, 0.0f, 0.0f};
                                    bf16x8_t pv;
                                    __builtin_memcpy(&pv, pw[a], 16);
                                    acc[m][a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(picks, pv, opens ? none : acc[m][a], 0, 0, 0);
                                } else if (q & 1) {
                                    if (half % HALVES == 0 && (q & 3) == 1) acc[m][a] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                                    bf16x16_t pv;
                                    __builtin_memcpy(&pv, pw[a], 32);
                                    acc[m][a] = __builtin_amdgcn_smfmac_f32_16x16x64_bf16(picks, pv, acc[m][a], places, 0, 0);
                                }
                            }
                            if (q + 1 < 16) d = ahead;
                            // Steps stay apart: left alone, the scheduler converts the first of the products
                            // ahead within this step and waits out the matrix instruction that makes them.
                            __builtin_amdgcn_sched_barrier(0);
                            if (half % HALVES == HALVES - 1 && (q & 7) == 7) fold();
                        }
                    }
                }
            }
            bool lost = false;
            if (v < r0) {
#pragma unroll
                for (int m = 0; m < 2; ++m)
#pragma unroll
                    for (int a = 0; a < 4; ++a) {
                        lost |= __builtin_isunordered(acc[m][a][0], acc[m][a][1]) |
                                __builtin_isunordered(acc[m][a][2], acc[m][a][3]);
                        u32x2 o;
                        o.x = f32x2_to_bf16x2(acc[m][a][0], acc[m][a][1]);
                        o.y = f32x2_to_bf16x2(acc[m][a][2], acc[m][a][3]);
                        org[(4 * m + a) * 64] = o;
                    }
                if (!CAREFUL && __any(lost)) {
                    at = {t0, v};
                    return false;
                }
                continue;
            }
            float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int m = 0; m < 2; ++m)
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    const u32x2 of = org[(4 * m + a) * 64];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const uint32_t o = h ? of.y : of.x;
                        const uint32_t cur = f32x2_to_bf16x2(acc[m][a][2 * h], acc[m][a][2 * h + 1]);
                        const uint32_t dd = f32x2_to_bf16x2(u2f(cur << 16) - u2f(o << 16),
                                                            u2f(cur & 0xFFFF0000u) - u2f(o & 0xFFFF0000u));
                        const float lo = u2f(dd << 16), hi = u2f(dd & 0xFFFF0000u);
                        sum[2 * h] += lo * lo;
                        sum[2 * h + 1] += hi * hi;
                    }
                }
            // a NaN output leaves a NaN here
            lost = __builtin_isunordered(sum[0], sum[1]) | __builtin_isunordered(sum[2], sum[3]);
            if (!CAREFUL && __any(lost)) {
                at = {t0, v};
                return false;
            }
            float total = (sum[0] + sum[1]) + (sum[2] + sum[3]);
            total += __shfl_xor(total, 32, kWave);   // the other tokens of the row
            const int r = row0 + fr;
            if (lane < 32 && r < n) loss[((int64_t)v * n + r) * nblk + b] += total / (float)tokens;
        }
    }
    return true;
}

// ------------------------------------------------------------------------------------- fp16
// A lane owns one row of one weight block, its quantised weights in registers, two a word; the
// activations are uniform over the wavefront (scalar loads, two columns a word).  One v_pk_mul_f16 gives
// two rounded products; the words of four tokens are summed as in the bf16 form, two steps of a chain an
// instruction: lane l, register i holds row l, token i of the four.  The partial outputs of the unclipped block stay in LDS.
template <int BS, bool CAREFUL>
__device__ __forceinline__ bool clip_losses_f16(const uint16_t* __restrict__ x, int tokens,
                                                const uint16_t* __restrict__ w, int n, int k,
                                                const void* __restrict__ w_amax, int amax_dtype,
                                                const ClipRatios& ratios, int r0, int r1, const IntOp& op,
                                                float* __restrict__ loss, u32x2* __restrict__ org, ClipStep& at) {
    constexpr int GW = 4;            // words of a token read ahead together (8 columns)
    constexpr int NG = BS / 2 / GW;
    constexpr int CHAINS = BS >= 32 ? 4 : 2;   // of sums, as independent as they are short
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nblk = k / BS, b = blockIdx.y;
    const int row0 = (blockIdx.x * kClipWaves + wave) * kClipLanes;
    if (row0 >= n) return true;
    org += (size_t)wave * (kClipTokens / 4) * kClipLanes + lane;
    const int row = row0 + lane < n ? row0 + lane : n - 1;
    const uint16_t* wp = w + (int64_t)row * k + b * BS;
    const float amax = load_scalar(w_amax, amax_dtype, (int64_t)row * nblk + b);
    f16x8_t picks;
    int places = 0;
    {
        uint32_t m[4];
        if constexpr (CAREFUL) clip_sum_operand(0x3C003C00u, m);
        else places = clip_sum_operand_sparse(0x3C003C00u, m);
        __builtin_memcpy(&picks, m, 16);
    }
    const uint32_t* xw = (const uint32_t*)(x + b * BS);
    const int xstride = k / 2;
    uint32_t wq[BS / 2];
    auto product = [](uint32_t xs, uint32_t ws) {   // of two pairs, each rounded
        f16x2_t a, c;
        __builtin_memcpy(&a, &xs, 4);
        __builtin_memcpy(&c, &ws, 4);
        const f16x2_t p = a * c;
        uint32_t out;
        __builtin_memcpy(&out, &p, 4);
        return out;
    };
    for (int t0 = CAREFUL ? __builtin_amdgcn_readfirstlane(at.token) : 0; t0 < tokens; t0 += kClipTokens) {
        const int tc = tokens - t0 < kClipTokens ? tokens - t0 : kClipTokens;
        for (int v = r0 - 1; v < r1; ++v) {   // r0 - 1: the unclipped block
            if (CAREFUL && v >= r0 && t0 == at.token && v < at.ratio) continue;   // in the losses already
            IntOp::Scale s = {};
            if (v >= r0) s = clip_scale(op, amax, amax_dtype, ratios.r[v]);
            // opaque to the optimiser, which would otherwise keep the block live beside its
            // quantised form instead of reading it again (L2) for every ratio
            const uint16_t* src = wp;
            asm volatile("" : "+v"(src));
#pragma unroll
            for (int c0 = 0; c0 < BS / 8; c0 += 2) {
                u32x4 raw[2] = {*(const u32x4*)(src + 8 * c0), *(const u32x4*)(src + 8 * c0 + 8)};
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const uint32_t rw[4] = {raw[c].x, raw[c].y, raw[c].z, raw[c].w};
                    float q[8];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        q[2 * j] = f16_bits_to_f32(rw[j] & 0xFFFFu);
                        q[2 * j + 1] = f16_bits_to_f32(rw[j] >> 16);
                    }
                    if (v >= r0) {
                        if (clip_fast(op, s)) {
#pragma unroll
                            for (int j = 0; j < 8; ++j) q[j] = clip_qdq_fast(op, q[j], s);
                        } else {
                            keep_branch();
#pragma unroll
                            for (int j = 0; j < 8; ++j) q[j] = op.apply<false>(q[j], s);
                        }
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            wq[4 * (c0 + c) + j] = f32_to_f16_bits(q[2 * j]) | (f32_to_f16_bits(q[2 * j + 1]) << 16);
                    } else {
#pragma unroll
                        for (int j = 0; j < 4; ++j) wq[4 * (c0 + c) + j] = rw[j];
                    }
                }
            }
            bool lost = false;
            float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            for (int g4 = 0; g4 * 4 < tc; ++g4) {
                const uint32_t* xr[4];   // past the end: the last token again, left out below
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int t = 4 * g4 + i < tc ? 4 * g4 + i : tc - 1;
                    xr[i] = xw + (int64_t)(t0 + t) * xstride;
                }
                f32x4 acc[CHAINS];
#pragma unroll
                for (int c = 0; c < CHAINS; ++c) acc[c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                auto sum_chains = [&]() {
                    f32x4 t = acc[0] + acc[1];
                    if constexpr (CHAINS == 4) t = t + (acc[2] + acc[3]);
                    return t;
                };
                f32x4 total;
                if constexpr (CAREFUL) {
                    uint32_t kind[4] = {0, 0, 0, 0};
#pragma unroll 1
                    for (int pass = 0; pass < 2; ++pass) {
                        #pragma unroll
                        for (int j = 0; j < BS / 2; ++j) {
                            // opaque, or the products would be kept from one pass for the other and the
                            // activations be read many steps ahead
                            int at_j = j;
                            asm volatile("" : "+s"(at_j));
                            uint32_t pw[4];
#pragma unroll
                            for (int i = 0; i < 4; ++i) pw[i] = clip_kinds_f16(product(xr[i][at_j], wq[j]), pass == 0);
                            f16x8_t pv;
                            __builtin_memcpy(&pv, pw, 16);
                            if (j < CHAINS) acc[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};   // of either pass
                            f32x4& c = acc[j % CHAINS];
                            c = __builtin_amdgcn_mfma_f32_16x16x32_f16(picks, pv, c, 0, 0, 0);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                        total = sum_chains();
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            if (pass == 0) kind[i] = clip_sum_kind(total[i]);
                            else total[i] = clip_with_kind(total[i], kind[i]);
                        }
                    }
                } else {
                    uint32_t pw[CHAINS][8];   // two steps of every chain
                    uint32_t cur[4][GW];
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int j = 0; j < GW; ++j) cur[i][j] = xr[i][j];
#pragma unroll
                    for (int g = 0; g < NG; ++g) {
                        uint32_t next[4][GW];
                        if (g + 1 < NG) {
#pragma unroll
                            for (int i = 0; i < 4; ++i)
#pragma unroll
                                for (int j = 0; j < GW; ++j) next[i][j] = xr[i][GW * (g + 1) + j];
                        }
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int j = 0; j < GW; ++j) {
                            const int step = GW * g + j, second = step / CHAINS & 1;
                            f32x4& c = acc[step % CHAINS];
                            uint32_t(&of)[8] = pw[step % CHAINS];
#pragma unroll
                            for (int i = 0; i < 4; ++i) of[4 * second + i] = product(cur[i][j], wq[step]);
                            if (second) {
                                f16x16_t pv;
                                __builtin_memcpy(&pv, of, 32);
                                c = __builtin_amdgcn_smfmac_f32_16x16x64_f16(picks, pv, c, places, 0, 0);
                            }
                        }
                        __builtin_amdgcn_sched_barrier(0);
                        if (g + 1 < NG) {
#pragma unroll
                            for (int i = 0; i < 4; ++i)
#pragma unroll
                                for (int j = 0; j < GW; ++j) cur[i][j] = next[i][j];
                        }
                    }
                    total = sum_chains();
                }
                float out[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) out[i] = clip_round<MO_F16>(total[i]);
                if (v < r0) {
                    lost |= __builtin_isunordered(total[0], total[1]) | __builtin_isunordered(total[2], total[3]);
                    u32x2 o;
                    o.x = f32_to_f16_bits(out[0]) | (f32_to_f16_bits(out[1]) << 16);
                    o.y = f32_to_f16_bits(out[2]) | (f32_to_f16_bits(out[3]) << 16);
                    org[g4 * kClipLanes] = o;
                } else {
                    const u32x2 o = org[g4 * kClipLanes];
                    const float og[4] = {f16_bits_to_f32(o.x & 0xFFFFu), f16_bits_to_f32(o.x >> 16),
                                         f16_bits_to_f32(o.y & 0xFFFFu), f16_bits_to_f32(o.y >> 16)};
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float d = clip_round<MO_F16>(out[i] - og[i]);
                        sum[i] += 4 * g4 + i < tc ? d * d : 0.0f;
                    }
                }
            }
            // a NaN output leaves a NaN here (a token past the end is the last one again)
            if (v >= r0) lost = __builtin_isunordered(sum[0], sum[1]) | __builtin_isunordered(sum[2], sum[3]);
            if (!CAREFUL && __any(lost)) {
                at = {t0, v};
                return false;
            }
            if (v < r0) continue;
            const float all = (sum[0] + sum[1]) + (sum[2] + sum[3]);
            if (row0 + lane < n) loss[((int64_t)v * n + row) * nblk + b] += all / (float)tokens;
        }
    }
    return true;
}

// ------------------------------------------------------------------------------------- fp32
// A lane owns one (output row, block), its quantised weights in registers; the activations of a token
// are uniform over the wavefront and are read through scalar loads; org[] of a lane lives in LDS
// ([token][lane], conflict-free).  A weight with few (row, block) pairs does not fill the chip with
// one wavefront per 64 pairs, so a workgroup may hold 2 wavefronts that own the same 64 pairs and
// share the tokens of a pass between them; their partial sums meet in LDS and wavefront 0 adds them in
// wavefront order, so the result does not depend on timing.
//
// For each of `tc` tokens, sum_j x[t, j] * w[j] in index order, handed to fn(t, value).  The scalar
// loads are software-pipelined one group of 16 elements ahead (across token boundaries too); they return
// out of order, so a wait covers every load in flight, hence the order "use the group that has
// arrived, then issue the next load, then do the vector work", which the scheduling barriers pin down.
template <int BS, typename Fn>
__device__ __forceinline__ void token_dots(const float* __restrict__ x, int64_t x0, int64_t stride,
                                           int tc, const float (&w)[BS], Fn fn) {
    constexpr int NG = BS / 16;
    const float* xp = x + x0;
    float cur[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) cur[j] = xp[j];
    for (int t = 0; t < tc; ++t) {
        const float* row = xp + (int64_t)t * stride;
        // the group after the last one of this token: the first of the next token (of this
        // token again after the last, a valid address whose data is not used)
        const float* next_row = t + 1 < tc ? row + stride : row;
        // four partial sums: the order of the fp32 accumulation is free, a single chain of
        // dependent adds is not
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            float xs[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) xs[j] = cur[j];
            __builtin_amdgcn_sched_barrier(0);
            const float* nxt = g + 1 < NG ? row + (g + 1) * 16 : next_row;
#pragma unroll
            for (int j = 0; j < 16; ++j) cur[j] = nxt[j];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < 16; ++j) acc[j & 3] += xs[j] * w[16 * g + j];
            __builtin_amdgcn_sched_barrier(0);
        }
        fn(t, (acc[0] + acc[1]) + (acc[2] + acc[3]));
    }
}

template <int BS>
__device__ __forceinline__ void clip_losses_f32(const float* __restrict__ x, int tokens,
                                                const float* __restrict__ w, int n, int k,
                                                const void* __restrict__ w_amax, int amax_dtype,
                                                const ClipRatios& ratios, int r0, int r1, const IntOp& op,
                                                float* __restrict__ loss, float* smem) {
    constexpr int NC = BS / 8;
    constexpr int GC = NC < 4 ? NC : 4;   // chunks loaded together
    // dynamic LDS: org[pass_tokens][64], then part[2][split][64]
    const int split = blockDim.x / kClipLanes;
    const int pass_tokens = split * kClipTokens;
    float (*org)[kClipLanes] = (float (*)[kClipLanes])smem;
    float (*part)[kClipLanes] = org + pass_tokens;
    const int lane = threadIdx.x % kClipLanes;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kClipLanes);
    const int nblk = k / BS;
    const int b = blockIdx.y;
    int row = blockIdx.x * kClipLanes + lane;
    const bool active = row < n;
    if (!active) row = n - 1;
    const int64_t w0 = (int64_t)row * k + (int64_t)b * BS;
    const int64_t xb = (int64_t)b * BS;
    const float amax = load_scalar(w_amax, amax_dtype, (int64_t)row * nblk + b);
    float wv[BS];
    // wv <- f(original block): the block is read again from memory (L2) every time, GC chunks
    // of loads in flight, rather than kept in a second set of registers
    auto refill = [&](auto f) {
        // opaque to the optimiser, or it would hoist the (loop-invariant) loads out of the
        // ratio loop and keep the whole block live in registers after all
        int64_t base = w0;
        asm volatile("" : "+v"(base));
#pragma unroll
        for (int c0 = 0; c0 < NC; c0 += GC) {
            RawChunk<MO_F32> raw[GC];
#pragma unroll
            for (int c = 0; c < GC; ++c) load_raw<MO_F32>(w, base + 8 * (c0 + c), raw[c]);
#pragma unroll
            for (int c = 0; c < GC; ++c) {
                float v[8];
                unpack_raw<MO_F32>(raw[c], v);
#pragma unroll
                for (int j = 0; j < 8; ++j) wv[8 * (c0 + c) + j] = f(v[j]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int flip = 0;   // part[] is double-buffered: one barrier per ratio is enough
    for (int t0 = 0; t0 < tokens; t0 += pass_tokens) {
        const int tc = tokens - t0 < pass_tokens ? tokens - t0 : pass_tokens;
        // this wavefront's share of the pass: tokens [lo, lo + mine)
        const int lo = (int)((int64_t)tc * wave / split);
        const int mine = (int)((int64_t)tc * (wave + 1) / split) - lo;
        const int64_t x0 = (int64_t)(t0 + lo) * k + xb;
        refill([](float v) { return v; });
        token_dots<BS>(x, x0, k, mine, wv, [&](int t, float v) { org[lo + t][lane] = v; });
        for (int r = r0; r < r1; ++r) {
            const IntOp::Scale s = clip_scale(op, amax, amax_dtype, ratios.r[r]);
            // the choice between the exact-reciprocal quotient and a division is per block, not
            // per element: one branch around the whole loop
            if (clip_fast(op, s)) refill([&](float v) { return clip_qdq_fast(op, v, s); });
            else refill([&](float v) { return op.apply<false>(v, s); });
            float sum = 0.0f;
            token_dots<BS>(x, x0, k, mine, wv, [&](int t, float cur) {
                const float d = cur - org[lo + t][lane];
                sum += d * d;
            });
            if (split > 1) {
                part[flip * split + wave][lane] = sum;
                __syncthreads();
                if (wave == 0) {
                    sum = part[flip * split][lane];
                    for (int v = 1; v < split; ++v) sum += part[flip * split + v][lane];
                }
                flip ^= 1;
            }
            if (active && wave == 0) {
                float* out = loss + ((int64_t)r * n + row) * nblk + b;
                *out += sum / (float)tokens;
            }
        }
    }
}

// blockIdx.z takes the ratios [z R / Z, (z + 1) R / Z): each share scores the unclipped block for itself
template <int DT, int BS>
__global__ __launch_bounds__(kClipLanes * kClipWaves, DT == MO_BF16 ? 3 : 2) void awq_clip_loss_kernel(
    const void* __restrict__ x, int tokens, const void* __restrict__ w, int n, int k,
    const void* __restrict__ w_amax, int amax_dtype, ClipRatios ratios, IntOp op,
    float* __restrict__ loss) {
    extern __shared__ __align__(16) unsigned char clip_smem[];
    const int r0 = (int)(blockIdx.z * (unsigned)ratios.count / gridDim.z);
    const int r1 = (int)((blockIdx.z + 1) * (unsigned)ratios.count / gridDim.z);
    if constexpr (DT == MO_BF16) {
        ClipStep at;
        // of a lane: 8 words of four partial sums, and 8 of four rounded outputs of the unclipped block
        f32x4* parts = (f32x4*)clip_smem + (threadIdx.x >> 6) * 512 + (threadIdx.x & 63);
        u32x2* org = (u32x2*)((f32x4*)clip_smem + kClipWaves * 512) + (threadIdx.x >> 6) * 512 + (threadIdx.x & 63);
        if (!clip_losses_bf16<BS, false>((const uint16_t*)x, tokens, (const uint16_t*)w, n, k, w_amax, amax_dtype,
                                         ratios, r0, r1, op, loss, parts, org, at))
            clip_losses_bf16<BS, true>((const uint16_t*)x, tokens, (const uint16_t*)w, n, k, w_amax, amax_dtype,
                                       ratios, r0, r1, op, loss, parts, org, at);
    } else if constexpr (DT == MO_F16) {
        ClipStep at;
        u32x2* org = (u32x2*)clip_smem;
        if (!clip_losses_f16<BS, false>((const uint16_t*)x, tokens, (const uint16_t*)w, n, k, w_amax, amax_dtype,
                                        ratios, r0, r1, op, loss, org, at))
            clip_losses_f16<BS, true>((const uint16_t*)x, tokens, (const uint16_t*)w, n, k, w_amax, amax_dtype,
                                      ratios, r0, r1, op, loss, org, at);
    } else
        clip_losses_f32<BS>((const float*)x, tokens, (const float*)w, n, k, w_amax, amax_dtype, ratios, r0, r1,
                            op, loss, (float*)clip_smem);
}

}  // namespace mo

// loss[r, row, b] += mean over tokens of the squared error of block (row, b) clipped at
// ratios[r] * w_amax[row, b]; see the header for the contract.
extern "C" int mo_awq_clip_losses(const void* x, int64_t tokens, const void* w, int64_t n,
                                  int64_t k, int dtype, int64_t block_size, const void* w_amax,
                                  int amax_dtype, const float* ratios, int n_ratios, int num_bits,
                                  int is_unsigned, int narrow_range, float* loss, void* stream) {
    if (tokens < 0 || n < 0 || k < 0 || n_ratios < 0) return MO_ERR_ARG;
    if (dtype < MO_F32 || dtype > MO_BF16) return MO_ERR_DTYPE;
    if (amax_dtype < MO_F32 || amax_dtype > MO_BF16) return MO_ERR_DTYPE;
    if (num_bits < 2 || num_bits > 16) return MO_ERR_ARG;
    if (block_size != 16 && block_size != 32 && block_size != 64 && block_size != 128)
        return MO_ERR_UNSUPPORTED;
    if (n_ratios > mo::kClipMaxRatios || k % block_size) return MO_ERR_UNSUPPORTED;
    if (tokens > 0x7FFFFFFF || n > 0x7FFFFFFF || k > 0x7FFFFFFF || k / block_size > 65535)
        return MO_ERR_UNSUPPORTED;
    if (tokens == 0 || n == 0 || k == 0 || n_ratios == 0) return MO_OK;
    if (!x || !w || !w_amax || !ratios || !loss) return MO_ERR_ARG;
    if ((((uintptr_t)x | (uintptr_t)w) & 15u) || ((uintptr_t)loss & 3u)) return MO_ERR_ARG;
    mo::ClipRatios rr;
    for (int i = 0; i < mo::kClipMaxRatios; ++i) rr.r[i] = i < n_ratios ? ratios[i] : 0.0f;
    rr.count = n_ratios;
    mo::IntOp op;
    op.bound = (float)((1 << (num_bits - 1 + (is_unsigned ? 1 : 0))) - 1);
    op.lo = is_unsigned ? 0.0f : (narrow_range ? -op.bound : -op.bound - 1.0f);
    const int rows_per_group = dtype == MO_BF16 ? 32 * mo::kClipWaves
                               : dtype == MO_F16 ? mo::kClipLanes * mo::kClipWaves : mo::kClipLanes;
    dim3 grid((unsigned)((n + rows_per_group - 1) / rows_per_group), (unsigned)(k / block_size));
    int waves = mo::kClipWaves;
    size_t smem = 0;
    if (dtype == MO_F32) {
        // Up to about 2048 sets of 64 pairs (two wavefronts per SIMD) two wavefronts to a set are
        // faster, from there on one is; each should still get 8 tokens or more, and org[] of a pass
        // stays within 64 KB of LDS.
        const int64_t sets = (int64_t)grid.x * grid.y;
        waves = sets < 2048 && tokens >= 16 ? 2 : 1;
        smem = (size_t)waves * mo::kClipTokens * mo::kClipLanes * 4 +
               (waves > 1 ? (size_t)2 * waves * mo::kClipLanes * sizeof(float) : 0);
    } else {
        smem = (size_t)mo::kClipWaves * mo::kClipLanes * (dtype == MO_F16 ? mo::kClipTokens * 2 : 8 * (16 + 8));
        // A wavefront goes through all ratios unless there are too few of them to fill the chip; then
        // 2 to 11 of them share the ratios, each scoring the unclipped block once more.  The lines lie where they were drawn
        // for dense sums; with sparse ones, 11 ratios, 64 tokens, blocks of 128, us by number of shares:
        //   bf16  4096 x 4096, 4096 wavefronts: 411, 433 with 2; 2048 x 4096, 2048: 211, 219 with 2; 1024 x 4096, 1024: 131, 117
        //         with 2, 119 with 3, 125 with 4; 1024 x 1024, 256: 129, 76 with 2, 45 with 4, 48 with 8
        //   fp16  4096 x 4096, 2048 wavefronts: 485, 443 with 2, 440 with 3, 462 with 4; 1024 x 4096, 512: 289, 142 with 4, 140 - 145
        //         with 6 (the line's), 159 with 8; 1024 x 1024, 128: 280, 98 with 4, 74 with 8, 67 with 11
        // The line is within 2 % of the best of them from 256 wavefronts on (blocks of 32 and 64 too); with fewer, bf16 would gain by
        // more than four shares (512 x 512, 64 wavefronts: 45 and 25 with 11).  Cards differ by some 8 %.
        // What bounds the bf16 form: a step of 2048 products is 96 cycles of matrix instructions (64 of products) and about
        // 90 of vector instructions (72 of conversions) plus 24 of the port that issues both; measured 160.  Higher
        // priority for the wavefront at its matrix instructions (402 us), sums between the conversions (424) or products
        // behind the first of them (444) win nothing.
        const int64_t sets = (int64_t)grid.x * grid.y * mo::kClipWaves;
        int64_t share = ((dtype == MO_BF16 ? 2048 : 3072) + sets - 1) / sets;
        if (dtype == MO_BF16 && share > 4) share = 4;
        if (share > n_ratios) share = n_ratios;
        grid.z = (unsigned)mo::tuned("clip_shares", share);
    }
    hipStream_t s = (hipStream_t)stream;
#define CALL(DT, BS)                                                                       \
    mo::awq_clip_loss_kernel<DT, BS><<<grid, mo::kClipLanes * waves, smem, s>>>(           \
        x, (int)tokens, w, (int)n, (int)k, w_amax, amax_dtype, rr, op, loss)
#define BY_BS(DT)                                                         \
    switch (block_size) {                                                 \
        case 16: CALL(DT, 16); break;                                     \
        case 32: CALL(DT, 32); break;                                     \
        case 64: CALL(DT, 64); break;                                     \
        default: CALL(DT, 128); break;                                    \
    }
    switch (dtype) {
        case MO_F32: BY_BS(MO_F32) break;
        case MO_F16: BY_BS(MO_F16) break;
        default: BY_BS(MO_BF16) break;
    }
#undef BY_BS
#undef CALL
    return hipGetLastError() == hipSuccess ? MO_OK : MO_ERR_LAUNCH;
}

namespace mo {
// The end of the search: per block the first smallest loss over the ratios (a NaN never wins, a block without a
// loss below infinity keeps a clip value of zero) and T(amax * ratio).  Reads each loss once; as tensor
// operations nine launches behind the search and its GEMM, 47 us for 11 x 131072 losses against 5.4.
template <int DT>
__global__ __launch_bounds__(256) void awq_best_clip_kernel(const float* __restrict__ loss, int n_ratios,
                                                            int64_t blocks, const float* __restrict__ ratios,
                                                            const void* __restrict__ amax,
                                                            float* __restrict__ best_loss, void* __restrict__ clip) {
    const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (b >= blocks) return;
    const float inf = __builtin_inff();
    float best = inf, ratio = 0.0f;
    for (int r = 0; r < n_ratios; ++r) {
        const float l = loss[r * blocks + b];
        const bool better = l < best;
        best = better ? l : best;
        ratio = better ? ratios[r] : ratio;
    }
    best_loss[b] = best;
    store_elem<DT>(clip, b, best < inf ? load_elem<DT>(amax, b) * ratio : 0.0f);
}
}  // namespace mo

extern "C" int mo_awq_best_clip(const float* loss, int64_t n_ratios, int64_t blocks, const float* ratios, const void* amax,
                                int dtype, float* best_loss, void* clip, void* stream) {
    if (n_ratios < 0 || n_ratios > 0x7FFFFFFF || blocks < 0) return MO_ERR_ARG;
    if (dtype < MO_F32 || dtype > MO_BF16) return MO_ERR_DTYPE;
    if (blocks == 0) return MO_OK;
    if (!best_loss || !clip || !amax || (n_ratios && (!loss || !ratios))) return MO_ERR_ARG;
    const int64_t g = (blocks + 255) / 256;
    if (g > 0x7FFFFFFF) return MO_ERR_UNSUPPORTED;
#define CALL(DT)                                                                                     \
    mo::awq_best_clip_kernel<DT><<<(unsigned)g, 256, 0, (hipStream_t)stream>>>(loss, (int)n_ratios, blocks, ratios, \
                                                                               amax, best_loss, clip)
    switch (dtype) {
        case MO_F32: CALL(MO_F32); break;
        case MO_F16: CALL(MO_F16); break;
        default: CALL(MO_BF16); break;
    }
#undef CALL
    return hipGetLastError() == hipSuccess ? MO_OK : MO_ERR_LAUNCH;
}
