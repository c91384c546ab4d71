// Row-wise fake quantisation for gfx950: x [rows, k] with rows of any length and alignment, optionally
// multiplied by one scale per column first -- what a quantizer with a pre-quant scale does to the input of
// a layer (SmoothQuant, AWQ) --, and the block formats and layouts that have no whole-tensor kernel.
//
// HBM-bound: one read and one write of the tensor.  Multiplying in a launch of its own moves the tensor
// twice as often.  A lane owns chunks of 8 columns of one row, all loads ahead of the first store; the
// scales of a chunk come from L2.  The product is rounded to the tensor's type before it is quantised, as
// the tensor expression rounds it.  Measured, each against the kernel it replaced: NVFP4 of fp16 1537 x 3000
// 7.0 us (15.4 with element loads and a division per element), INT8 of a scaled bf16 2048 x 14336 22.7 us
// (43.2 with the product in a launch of its own), NVFP4 of fp32 4096 x 8192 53 us (69), MX E4M3 of
// bf16 3001 x 5001 15 us (43 with element loads) and of 8192 x 8192 43 us (47).  Without a scale and aligned
// it equals the whole-tensor kernels or beats them at most sizes; whole_is_faster says where it does not.
#include "common.h"
#include "blockfp_ops.h"
#include "nvfp4_ops.h"
#include "qdq_ops.h"

namespace mo {

// Chunks of 8 elements per lane.  8192 x 8192 bf16, MX E4M3: 43.2 us = 6.2 TB/s with two, 44.3 with one and
// 45.7 with four; with a scale per column 46.5, 48.2 and 49.4 (an occupancy cap moves nothing by more than
// 1 %, with one chunk it costs 10 %).
constexpr int kRowU = 2;
constexpr int kRowTileChunks = 256 * kRowU;

template <int DT>
__device__ __forceinline__ float row_round(float v) {
    if constexpr (DT == MO_BF16) return round_to_bf16(v);
    else if constexpr (DT == MO_F16) return f16_bits_to_f32(f32_to_f16_bits(v));
    else return v;
}

// The formats: `start` once per lane, `chunk` for 8 elements (zeros where the row has ended).
template <bool SAT>
struct RowFp8 {
    Fp8Op<true> op;
    Fp8Op<true>::Scale s;
    __device__ __forceinline__ void start(float amax) { s = op.make(amax); }
    template <int DT>
    __device__ __forceinline__ void chunk(const float (&v)[8], float (&o)[8]) const {
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
            o[j] = v[j];
            o[j + 1] = v[j + 1];
            op.template apply2<SAT>(o[j], o[j + 1], s, s);
        }
    }
};

struct RowInt {
    IntOp op;
    IntOp::Scale s;
    __device__ __forceinline__ void start(float amax) { s = op.make(amax); }
    template <int DT>
    __device__ __forceinline__ void chunk(const float (&v)[8], float (&o)[8]) const {
        if (s.fast) {
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = op.apply_fast<false>(v[j], s);
        } else {
            keep_branch();
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = op.apply<false>(v[j], s);
        }
    }
};

template <int BS, int MODE>
struct RowNvfp4 {
    static constexpr int lanes_lg = BS == 8 ? 0 : (BS == 16 ? 1 : 2);   // lanes that share a block, as a power of two
    float gs, gs_safe;
    __device__ __forceinline__ void start(float amax) {
        gs = amax / 2688.0f;
        gs_safe = gs > 0.0f ? gs : 1e-12f;
    }
    template <int DT>
    __device__ __forceinline__ void chunk(const float (&v)[8], float (&o)[8]) const {
        const uint32_t m = group_max_u32(chunk_absmax_bits(v), lanes_lg);
        nvfp4_qdq_chunk<DT, MODE>(v, m, nvfp4_unit<MODE>(u2f(m), gs, gs_safe), o);
    }
};

template <int FMT>
struct RowMx {   // power-of-two block scales
    int lg;
    __device__ __forceinline__ void start(float) {}
    template <int DT>
    __device__ __forceinline__ void chunk(const float (&v)[8], float (&o)[8]) const {
        const uint32_t m = group_max_u32(block_fp_absmax(v), lg);
        block_fp_chunk<FMT>(v, block_scale<FMT>(u2f(m), MO_EF_E8M0, false, 0.0f), o);
    }
};

template <int DT, typename F>
__global__ __launch_bounds__(256) void row_qdq_kernel(const void* __restrict__ x, void* __restrict__ y,
                                                      uint32_t chunks, int64_t k, RowDiv div,
                                                      const void* __restrict__ pre,
                                                      const void* __restrict__ amax, int amax_dtype, F f) {
    __shared__ uint32_t smem[4];
    f.start(amax ? tensor_amax(amax, amax_dtype, smem) : 0.0f);
    const uint32_t c0 = blockIdx.x * kRowTileChunks + threadIdx.x;
    RawChunk<DT> raw[kRowU], sc[kRowU];
    uint32_t row[kRowU], col[kRowU];
#pragma unroll
    for (int u = 0; u < kRowU; ++u) {
        uint32_t c = c0 + u * 256;
        c = c < chunks ? c : chunks - 1;
        row[u] = row_of(c, div);
        col[u] = (c - row[u] * div.d) << 3;
        load_raw_row<DT>(x, (int64_t)row[u] * k, col[u], k, raw[u]);
    }
    if (pre) {
#pragma unroll
        for (int u = 0; u < kRowU; ++u) load_raw_row<DT>(pre, 0, col[u], k, sc[u]);
    }
#pragma unroll
    for (int u = 0; u < kRowU; ++u) {
        float v[8], o[8];
        unpack_raw<DT>(raw[u], v);
        if (pre) {
            float s[8];
            unpack_raw<DT>(sc[u], s);
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = row_round<DT>(v[j] * s[j]);
        }
        f.template chunk<DT>(v, o);
        if (c0 + u * 256 < chunks) store_row<DT>(y, (int64_t)row[u] * k, col[u], k, o);
    }
}

template <int DT, typename F>
static void launch_row(const void* x, void* y, int64_t rows, int64_t k, int64_t block, const void* pre,
                       const void* amax, int amax_dtype, F f, hipStream_t s) {
    const int64_t cpr = (k + block - 1) / block * (block / 8);
    constexpr int64_t kMost = 1ll << 27;   // chunks of a launch: chunk and column numbers stay within 32 bits
    if (cpr > kMost) {                     // rows of a gigabyte: piece by piece, whole blocks
        for (int64_t r = 0; r < rows; ++r)
            for (int64_t c = 0; c < k; c += kMost * 8) {
                const int64_t off = (r * k + c) * Elem<DT>::bytes;
                launch_row<DT, F>((const char*)x + off, (char*)y + off, 1, k - c < kMost * 8 ? k - c : kMost * 8, block,
                                  pre ? (const char*)pre + c * Elem<DT>::bytes : nullptr, amax, amax_dtype, f, s);
            }
        return;
    }
    const RowDiv div = row_div((uint32_t)cpr);
    const int64_t step = kMost / cpr;
    for (int64_t r0 = 0; r0 < rows; r0 += step) {
        const int64_t here = rows - r0 < step ? rows - r0 : step, chunks = here * cpr;
        const int64_t off = r0 * k * Elem<DT>::bytes;
        row_qdq_kernel<DT, F><<<(unsigned)((chunks + kRowTileChunks - 1) / kRowTileChunks), 256, 0, s>>>(
            (const char*)x + off, (char*)y + off, (uint32_t)chunks, k, div, pre, amax, amax_dtype, f);
    }
}

template <int DT>
static int dispatch_row(const void* x, void* y, int64_t rows, int64_t k, const void* pre, int kind, int p0, int p1,
                        int p2, const void* amax, int amax_dtype, hipStream_t s) {
    const int64_t block = kind == MO_ROW_NVFP4 || kind == MO_ROW_MX ? p0 : 8;
#define RUN(...) launch_row<DT>(x, y, rows, k, block, pre, amax, amax_dtype, __VA_ARGS__, s)
    if (kind == MO_ROW_FP8) {
        if (p0) RUN(RowFp8<true>{}); else RUN(RowFp8<false>{});
    } else if (kind == MO_ROW_INT) {
        RowInt f = {};
        f.op.bound = (float)((1 << (p0 - 1 + (p1 ? 1 : 0))) - 1);
        f.op.lo = p1 ? 0.0f : (p2 ? -f.op.bound : -f.op.bound - 1.0f);
        RUN(f);
    } else if (kind == MO_ROW_NVFP4) {
        if (p0 == 8) { if (p1) RUN(RowNvfp4<8, 1>{}); else RUN(RowNvfp4<8, 0>{}); }
        else if (p0 == 16) { if (p1) RUN(RowNvfp4<16, 1>{}); else RUN(RowNvfp4<16, 0>{}); }
        else { if (p1) RUN(RowNvfp4<32, 1>{}); else RUN(RowNvfp4<32, 0>{}); }
    } else {
        const int lg = p0 == 8 ? 0 : (p0 == 16 ? 1 : 2);
        switch (p1) {
#define MX(F) case F: RUN(RowMx<F>{lg}); break;
            MX(MO_EF_E4M3) MX(MO_EF_E5M2) MX(MO_EF_INT8) MX(MO_EF_E0M3) MX(MO_EF_E1M2) MX(MO_EF_E3M0)
            MX(MO_EF_E2M1) MX(MO_EF_E3M2) MX(MO_EF_E2M3)
#undef MX
        }
    }
#undef RUN
    return MO_OK;
}

static int check_row_format(int kind, int p0, int p1) {
    const bool block = p0 == 8 || p0 == 16 || p0 == 32;
    switch (kind) {
        case MO_ROW_INT: return p0 < 1 || p0 > 24 ? MO_ERR_ARG : MO_OK;
        case MO_ROW_FP8: return MO_OK;
        case MO_ROW_NVFP4:
            if (p1 != 0 && p1 != 1) return MO_ERR_ARG;
            return block ? MO_OK : MO_ERR_UNSUPPORTED;
        case MO_ROW_MX: return !block || p1 < MO_EF_E4M3 || p1 > MO_EF_E2M3 ? MO_ERR_UNSUPPORTED : MO_OK;
        default: return MO_ERR_UNSUPPORTED;
    }
}

// Where rows do not matter (no scale per column, 16-byte alignment, one amax at hand) and the kernels for whole
// tensors are the faster ones.  A workgroup of theirs takes twice the chunks, so from 2^23 to 2^24 elements they fill
// the chip in one round where the row kernel starts a second: bf16 32 MB FP8 11.1 us against 12.2, INT8 11.7 and
// 12.0, fp16 11.5 and 12.5, 11.5 and 12.7.  In fp16, whose conversions cost the row kernel more, from 2^20 (4 MB
// 3.6 and 3.8; 16 MB 7.0 and 6.9), and in fp32 as long as the tensor is below 1 GB (16 MB 7.4 and 7.3, 32 MB 13.8 and
// 14.7, 128 MB 51.3 and 52.5, 512 MB 204 and 204, 1 GB 410 and 419, 4 GB 1737 and 1715).  Elsewhere the row kernel is equal or
// faster (bf16 INT8 1 MB 3.2 and 2.7, 256 MB 86.6 and 82.4, FP8 84.5 and 83.4).  Same bits either way.
static bool whole_is_faster(int64_t n, int dtype) {
    if (dtype == MO_F32) return n >= (1ll << 22) && n <= (1ll << 28);
    return n > (dtype == MO_F16 ? 1ll << 20 : 1ll << 23) && n <= (1ll << 24);
}

// amax_dtype: a type, or parts (kAmaxParts + their number)
int row_qdq(const void* x, void* y, int64_t rows, int64_t k, int dtype, const void* pre, int kind, int p0, int p1,
            int p2, const void* amax, int amax_dtype, hipStream_t s) {
    int rc;
    if (!pre && amax_dtype < kAmaxParts) {
        const int64_t n = rows * k;
        const bool aligned = (((uintptr_t)x | (uintptr_t)y) & 15u) == 0;
        if (kind == MO_ROW_FP8 && aligned && whole_is_faster(n, dtype))
            return mo_fp8_qdq(x, y, 1, 1, n, dtype, amax, amax_dtype, p0, s);
        if (kind == MO_ROW_INT && aligned && whole_is_faster(n, dtype))
            return mo_int_qdq(x, y, 1, 1, n, dtype, amax, amax_dtype, p0, p1, p2, s);
        if (kind == MO_ROW_NVFP4) {
            rc = nvfp4_qdq_whole(x, y, n, k, dtype, p0, p1, amax, amax_dtype, s);
            if (rc != MO_ERR_UNSUPPORTED) return rc;
        }
    }
    switch (dtype) {
        case MO_F32: rc = dispatch_row<MO_F32>(x, y, rows, k, pre, kind, p0, p1, p2, amax, amax_dtype, s); break;
        case MO_F16: rc = dispatch_row<MO_F16>(x, y, rows, k, pre, kind, p0, p1, p2, amax, amax_dtype, s); break;
        default: rc = dispatch_row<MO_BF16>(x, y, rows, k, pre, kind, p0, p1, p2, amax, amax_dtype, s); break;
    }
    if (rc != MO_OK) return rc;
    return hipGetLastError() == hipSuccess ? MO_OK : MO_ERR_LAUNCH;
}

}  // namespace mo

extern "C" int mo_row_qdq(const void* x, void* y, int64_t rows, int64_t k, int dtype, const void* pre_scale,
                          int kind, int p0, int p1, int p2, const void* amax, int amax_dtype, void* stream) {
    if (rows < 0 || k < 0) return MO_ERR_ARG;
    if (dtype < MO_F32 || dtype > MO_BF16 || amax_dtype < MO_F32 || amax_dtype > MO_BF16) return MO_ERR_DTYPE;
    const int format = mo::check_row_format(kind, p0, p1);
    if (format != MO_OK) return format;
    if (rows == 0 || k == 0) return MO_OK;
    if (!x || !y || (kind != MO_ROW_MX && !amax)) return MO_ERR_ARG;
    const uintptr_t need = dtype == MO_F32 ? 3u : 1u;
    if (((uintptr_t)x | (uintptr_t)y | (uintptr_t)pre_scale) & need) return MO_ERR_ARG;
    return mo::row_qdq(x, y, rows, k, dtype, pre_scale, kind, p0, p1, p2, amax, amax_dtype, (hipStream_t)stream);
}

// The abs-max parts and the fake quantisation that folds them: two launches, nothing to clear.
// 4096 x 4096 bf16 to FP8: 18.9 us, 33.2 as four launches (fill, abs-max, conversion, quantise).
extern "C" int mo_dynamic_qdq(const void* x, void* y, int64_t rows, int64_t k, int dtype, int kind, int p0, int p1,
                              int p2, void* parts, void* stream) {
    if (rows < 0 || k < 0) return MO_ERR_ARG;
    if (dtype < MO_F32 || dtype > MO_BF16) return MO_ERR_DTYPE;
    const int format = kind == MO_ROW_MX ? MO_ERR_UNSUPPORTED : mo::check_row_format(kind, p0, p1);
    if (format != MO_OK) return format;
    if (rows == 0 || k == 0) return MO_OK;
    if (!x || !y || !parts) return MO_ERR_ARG;
    if (((uintptr_t)x | (uintptr_t)y) & 15u) return MO_ERR_UNSUPPORTED;
    hipStream_t s = (hipStream_t)stream;
    int nparts = 0;
    const int rc = mo::launch_absmax_parts(x, rows * k, dtype, true, (uint32_t*)parts, &nparts, s);
    if (rc != MO_OK) return rc;
    return mo::row_qdq(x, y, rows, k, dtype, nullptr, kind, p0, p1, p2, parts, mo::kAmaxParts + nparts, s);
}
