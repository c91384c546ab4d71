// Input gradient of a linear layer with a fake-quantised weight, for gfx950:
//
//   dx[t, k] = T(sum over n of dy[t, n] * wq[n, k])
//
// A training step has a few hundred tokens, so the result is small, the weight is read once and the sum is long: the
// result alone has too few tiles for 256 compute units, and the sum over n is cut into runs whose fp32 partial sums a
// second launch adds in order (one rounding, the same bits on every call).
//
// 64, 128 or 256 tokens x 128 columns a workgroup, 64 n a step.  The gradient is contiguous along the sum, as the
// matrix instructions want it; the weight is not, and gfx950 turns it on the way out of LDS (ds_read_b64_tr_b16: 16
// lanes read 4 n of 16 columns, each lane gets 4 n of one).  Three LDS stages: one is multiplied, the next is
// complete, so that the first operands of a step are read before its barrier, and the loads of the one after that are
// written to LDS between the products; global loads run two steps further ahead, in registers.  Loads go through
// buffer descriptors that end with the run of n: tokens and n past an edge read as zero.  Columns past the edge of k read the
// start of the next row, and belong to results that are not stored.
//
// Measured against the library's product, bf16, weight 14336 x 4096 (n x k): 32 tokens 22.7 us (41.8), 128 28.1 (96.8),
// 256 44.7 (76.8), 512 72.5 (100 - 110) = 0.83 PFLOP/s, 1024 128 (147).  Up to 128 tokens memory bounds it (117 MB of weight, 4.2 - 5.2 TB/s with
// the second launch); beyond, the matrix cores are busy 40 % of the cycles (512 tokens): a step's 1024 cycles of
// products stand beside 910 of LDS and 768 of L1 (64 bytes a clock), and with no loads at all 512 tokens x 4096 x 14336
// take 55 us where they take 66 with them.  Operands read three products ahead 66.0, two 66.9, one 67.7; two LDS stages 73.
// No bank conflicts (counted).
#include "mfma_ops.h"

namespace mo {

constexpr int kDgCols = 128;     // results of a workgroup along k
constexpr uint32_t kDgSplits = 16;   // most runs that the sum over n is cut into
constexpr int kDgStep = 64;      // n of a step
constexpr int kAhead = 3;        // of the four products of a step, how far ahead their operands are read

// Byte offset of 8 columns of n of a token in its tile (128 bytes a token)
__device__ __forceinline__ int dgrad_dy_slot(int row, int octet) {
    return row * 128 + ((octet ^ row ^ (row >> 3)) & 7) * 16;
}
// Byte offset of 8 columns of k of an n in the weight's tile (256 bytes an n)
__device__ __forceinline__ int dgrad_w_slot(int row, int octet) {
    return row * 256 + ((octet ^ (row << 2)) & 15) * 16;
}

// WM x 2 wavefronts, 32 * MI tokens x 64 columns each
template <int DT, int WM, int MI>
__global__ __launch_bounds__(WM * 128, 2) void dgrad_kernel(
    const uint16_t* __restrict__ dy, const uint16_t* __restrict__ w, uint16_t* __restrict__ dx,
    float* __restrict__ partial, uint32_t tokens, uint32_t n_all, uint32_t k_all, uint32_t tiles_t,
    uint32_t tiles_k, uint32_t splits, uint32_t steps) {
    constexpr int kThreads = WM * 128, kRows = WM * MI * 32;
    constexpr int kA = kRows * 8 / kThreads, kB = kDgStep * 16 / kThreads;   // chunks of a lane
    constexpr int kABytes = kRows * 128, kStage = kABytes + kDgStep * 256;
    __shared__ __align__(16) uint8_t lds[3 * kStage];

    const uint32_t id = xcd_tile(tiles_t * tiles_k * splits);
    const uint32_t t0 = id % tiles_t * kRows, rem = id / tiles_t, k0 = rem % tiles_k * kDgCols;
    const uint32_t split = rem / tiles_k;
    const uint32_t first = (uint32_t)((uint64_t)steps * split / splits);
    const uint32_t last = (uint32_t)((uint64_t)steps * (split + 1) / splits);
    const uint32_t n_end = last * kDgStep < n_all ? last * kDgStep : n_all;

    const auto dy_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)dy, 0, (int)(tokens * n_all * 2), 0x00020000);
    const auto w_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)w, 0, (int)(n_end * k_all * 2), 0x00020000);

    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint32_t a_off[kA], b_off[kB];
    int a_dst[kA], b_dst[kB];
    uint32_t a_n = first * kDgStep + (tid & 7) * 8;
#pragma unroll
    for (int i = 0; i < kA; ++i) {
        const uint32_t row = (i * kThreads + tid) >> 3;
        a_off[i] = ((t0 + row) * n_all + a_n) * 2;
        a_dst[i] = dgrad_dy_slot(row, tid & 7);
    }
#pragma unroll
    for (int i = 0; i < kB; ++i) {
        const uint32_t row = (i * kThreads + tid) >> 4;
        b_off[i] = ((first * kDgStep + row) * k_all + k0 + (tid & 15) * 8) * 2;
        b_dst[i] = kABytes + dgrad_w_slot(row, tid & 15);
    }
    struct Stage { u32x4 a[kA], b[kB]; };
    auto load = [&](Stage& r) {
        const bool in = a_n < n_end;
#pragma unroll
        for (int i = 0; i < kA; ++i) {
            r.a[i] = __builtin_amdgcn_raw_buffer_load_b128(dy_rsrc, in ? a_off[i] : 0xFFFFFFF0u, 0, 0);
            a_off[i] += kDgStep * 2;
        }
#pragma unroll
        for (int i = 0; i < kB; ++i) {
            r.b[i] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, b_off[i], 0, 0);
            b_off[i] += kDgStep * k_all * 2;
        }
        a_n += kDgStep;
    };
    // chunks [from, to) of a lane, those of dy first
    auto store = [&](const Stage& r, int at, int from, int to) {
#pragma unroll
        for (int i = 0; i < kA + kB; ++i)
            if (i >= from && i < to) {
                if (i < kA) *(u32x4*)(lds + at + a_dst[i < kA ? i : 0]) = r.a[i < kA ? i : 0];
                else *(u32x4*)(lds + at + b_dst[i < kA ? 0 : i - kA]) = r.b[i < kA ? 0 : i - kA];
            }
    };

    const int l32 = lane & 31, half = lane >> 5;
    const int wt = (wave >> 1) * MI * 32, wk = (wave & 1) * 64;
    int w_at[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int row = half * 8 + ((lane & 15) >> 2), col = wk + i * 32 + ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
        w_at[i] = kABytes + dgrad_w_slot(row, col >> 3) + (col & 4) * 2;
    }
    f32x16 acc[2][MI];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < MI; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    struct Operands { u32x4 a[2], b[MI]; };
    auto read = [&](Operands& f, int at, int s) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const u32x2 lo = lds_transposed(lds + at + w_at[i] + s * 16 * 256);
            const u32x2 hi = lds_transposed(lds + at + w_at[i] + (s * 16 + 4) * 256);
            f.a[i] = u32x4{lo.x, lo.y, hi.x, hi.y};
        }
#pragma unroll
        for (int j = 0; j < MI; ++j) f.b[j] = *(const u32x4*)(lds + at + dgrad_dy_slot(wt + j * 32 + l32, 2 * s + half));
    };
    auto multiply = [&](const Operands& f) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < MI; ++j) acc[i][j] = mfma_32x32x16<DT>(f.a[i], f.b[j], acc[i][j]);
    };

    const uint32_t count = last - first;
    int now = 0, next = kStage, after = 2 * kStage;   // LDS stages: multiplied, complete, being written
    Operands f[4];
    // One step: r holds the step after the next, and then the loads of the second one behind that
    auto step = [&](Stage& r) {
        constexpr int kPart = (kA + kB + 2) / 3;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if (s + kAhead < 4) read(f[(s + kAhead) & 3], now, s + kAhead);
            else read(f[(s + kAhead) & 3], next, s + kAhead - 4);
            if (s < 3) store(r, after, s * kPart, (s + 1) * kPart);
            else load(r);
            multiply(f[s]);
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
        const int free = now;
        now = next;
        next = after;
        after = free;
    };
    Stage r0, r1;
    load(r0);
    load(r1);
    store(r0, now, 0, kA + kB);
    load(r0);
    store(r1, next, 0, kA + kB);
    load(r1);
    __syncthreads();
#pragma unroll
    for (int s = 0; s < kAhead; ++s) read(f[s], now, s);
    for (uint32_t s = 0; s < count; s += 2) {   // steps past the end are zeros
        step(r0);
        step(r1);
    }

#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < MI; ++j) {
            const uint32_t t = t0 + wt + j * 32 + l32;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const uint32_t k = k0 + wk + i * 32 + g * 8 + half * 4;
                if (t >= tokens || k >= k_all) continue;
                const f32x16 v = acc[i][j];
                if (splits > 1) {
                    f32x4 o = {v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]};
                    *(f32x4*)(partial + ((size_t)split * tokens + t) * k_all + k) = o;
                } else {
                    u32x2 o;
                    o.x = round_pair<DT>(v[4 * g], v[4 * g + 1]);
                    o.y = round_pair<DT>(v[4 * g + 2], v[4 * g + 3]);
                    *(u32x2*)(dx + (size_t)t * k_all + k) = o;
                }
            }
        }
}

template <int DT>
__global__ __launch_bounds__(256) void dgrad_sum_kernel(const float* __restrict__ partial, uint16_t* __restrict__ dx,
                                                        size_t chunks, uint32_t splits) {
    const size_t c = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= chunks) return;
    f32x4 lo = {0, 0, 0, 0}, hi = {0, 0, 0, 0};
    const f32x4* p = (const f32x4*)partial + c * 2;
#pragma unroll 4
    for (uint32_t s = 0; s < splits; ++s, p += chunks * 2) {
        const f32x4 a = p[0], b = p[1];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            lo[j] += a[j];
            hi[j] += b[j];
        }
    }
    u32x4 o;
    o.x = round_pair<DT>(lo[0], lo[1]);
    o.y = round_pair<DT>(lo[2], lo[3]);
    o.z = round_pair<DT>(hi[0], hi[1]);
    o.w = round_pair<DT>(hi[2], hi[3]);
    *(u32x4*)(dx + c * 8) = o;
}

struct DgradPlan { int wm, mi; uint32_t tiles_t, tiles_k, splits, steps; };

// The tile and the runs of n with the least estimated time (us): every compute unit takes one workgroup after another, a
// step of 64 n takes 0.42, 0.6 and 1.03 in tiles of 64, 128 and 256 tokens, a workgroup 5 beside its steps; partial
// sums cost a launch and two passes over them.  In a sweep of 66 shapes (32 to 1024 tokens) the choice was within 5 % of the
// best for 57 and within 13 % for the rest, which take 8 to 20 us.
static DgradPlan dgrad_plan(int64_t tokens, int64_t n, int64_t k) {
    constexpr struct { int wm, mi; double step; } kTiles[] = {{2, 1, 0.42}, {4, 1, 0.6}, {4, 2, 1.03}};
    DgradPlan best{};
    double least = 0;
    for (const auto& tile : kTiles) {
        DgradPlan p{tile.wm, tile.mi, 0, 0, 1, 0};
        const int64_t rows = tile.wm * tile.mi * 32;
        p.tiles_t = (uint32_t)((tokens + rows - 1) / rows);
        p.tiles_k = (uint32_t)((k + kDgCols - 1) / kDgCols);
        p.steps = (uint32_t)((n + kDgStep - 1) / kDgStep);
        const uint64_t tiles = (uint64_t)p.tiles_t * p.tiles_k;
        for (uint32_t s = 1; s <= kDgSplits && s <= p.steps; ++s) {
            const double rounds = (double)((tiles * s + 255) / 256), each = (p.steps + s - 1) / s;
            double us = rounds * (each * tile.step + 5);
            if (s > 1) us += 3 + 1e-6 * s * tokens * k;
            if (least == 0 || us < least) {
                least = us;
                best = p;
                best.splits = s;
            }
        }
    }
    return best;
}

}  // namespace mo

static bool dgrad_takes(int64_t tokens, int64_t n, int64_t k) {
    if (tokens <= 0 || n <= 0 || k <= 0 || n % 8 || k % 8) return false;
    const int64_t limit = 0x7FFFFFFF;   // 32-bit byte offsets, of the loads past the last run too
    return tokens <= 65536 && (tokens + 256) * n * 2 <= limit && (n + 512) * k * 2 <= limit;
}

extern "C" int mo_input_grad_splits(int64_t tokens, int64_t n, int64_t k) {
    return dgrad_takes(tokens, n, k) ? (int)mo::dgrad_plan(tokens, n, k).splits : 0;
}

extern "C" int mo_input_grad_tile(int64_t tokens, int64_t n, int64_t k) {
    if (!dgrad_takes(tokens, n, k)) return 0;
    const mo::DgradPlan p = mo::dgrad_plan(tokens, n, k);
    return p.wm * p.mi * 32;
}

extern "C" int mo_input_grad(const void* dy, const void* w, void* dx, float* partial, int64_t tokens, int64_t n,
                             int64_t k, int dtype, int splits, void* stream) {
    if (tokens < 0 || n < 0 || k < 0) return MO_ERR_ARG;
    if (dtype < MO_F32 || dtype > MO_BF16) return MO_ERR_DTYPE;
    if (dtype == MO_F32) return MO_ERR_UNSUPPORTED;
    if (tokens == 0 || k == 0) return MO_OK;
    if (!dgrad_takes(tokens, n, k)) return MO_ERR_UNSUPPORTED;
    if (!dy || !w || !dx || splits < 1 || splits > (int)mo::kDgSplits || (splits > 1 && !partial)) return MO_ERR_ARG;
    if (((uintptr_t)dy | (uintptr_t)w | (uintptr_t)dx | (uintptr_t)partial) & 15u) return MO_ERR_UNSUPPORTED;
    mo::DgradPlan p = mo::dgrad_plan(tokens, n, k);
    p.splits = (uint32_t)splits;
    if (p.splits > p.steps) return MO_ERR_ARG;
    hipStream_t s = (hipStream_t)stream;
#define CALL(DT, WM, MI)                                                                                       \
    mo::dgrad_kernel<DT, WM, MI><<<p.tiles_t * p.tiles_k * p.splits, WM * 128, 0, s>>>(                        \
        (const uint16_t*)dy, (const uint16_t*)w, (uint16_t*)dx, partial, (uint32_t)tokens, (uint32_t)n,        \
        (uint32_t)k, p.tiles_t, p.tiles_k, p.splits, p.steps)
#define PICK(DT)                                                                                               \
    if (p.mi == 2) CALL(DT, 4, 2); else if (p.wm == 4) CALL(DT, 4, 1); else CALL(DT, 2, 1)
    if (dtype == MO_BF16) { PICK(MO_BF16); } else { PICK(MO_F16); }
#undef PICK
#undef CALL
    if (p.splits > 1) {
        const size_t chunks = (size_t)tokens * k / 8;
        const unsigned blocks = (unsigned)((chunks + 255) / 256);
        if (dtype == MO_BF16) mo::dgrad_sum_kernel<MO_BF16><<<blocks, 256, 0, s>>>(partial, (uint16_t*)dx, chunks, p.splits);
        else mo::dgrad_sum_kernel<MO_F16><<<blocks, 256, 0, s>>>(partial, (uint16_t*)dx, chunks, p.splits);
    }
    return hipGetLastError() == hipSuccess ? MO_OK : MO_ERR_LAUNCH;
}
