// gemm.hip — the batched product gemm_quant (kernels.cpp:289-345) on gfx950.
//
// y[t][o] = dot(dequantize_row(W row o), x_t) for every token t: the row is
// dequantised exactly (dequantize_row, quant.cpp:163-318) and each dot is the
// reference's dot_avx2 (kernels.cpp:206-223): two 8-lane FMA chains (k mod 16
// < 8 and >= 8), their sum, the 8-lane tree, then an FMA tail. Every output is
// the reference's bit for bit.
//
// A workgroup owns 32 weight rows x 32 or 64 tokens and runs the chains on
// the f32 matrix cores (chain_mfma.hpp). The K loop stages 64 columns at a
// time in one of two LDS buffers: the 32 rows dequantised from their raw
// blocks (8 elements per thread) and the tokens' inputs, both requested from
// memory a stage ahead, so that a stage costs one barrier.
#include "chain_mfma.hpp"
#include "fmx_internal.hpp"

#include <type_traits>

namespace fmx {

namespace {

constexpr uint32_t kGmRows = 32; // weight rows per workgroup
constexpr uint32_t kGmK = 64;    // columns per stage
constexpr uint32_t kGmStride = cm_stride<kGmK>();

// Loads of any alignment: raw blocks are only 2-byte aligned within a row.
typedef unsigned int gm_u32 __attribute__((aligned(1)));
typedef unsigned short gm_u16 __attribute__((aligned(1)));
typedef unsigned int gm_u32x2 __attribute__((ext_vector_type(2), aligned(1)));
typedef unsigned int gm_u32x4 __attribute__((ext_vector_type(4), aligned(1)));
typedef float gm_f32x4 __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ float ubyte_f32(uint32_t w, int b) { return static_cast<float>((w >> (8 * b)) & 0xFFu); }

// Elements e .. e + 7 (e a multiple of 8) of a raw row: load() requests their
// bytes, decode() forms the values by the expressions of the block
// dequantiser (quant.hip), so they are the reference's exactly. held() makes
// the loaded words opaque where it stands: without it the compiler moves the
// decoding's first shifts up to the load, across the loop, and waits there
// for a request that was meant to stay in flight for several stages.
__device__ __forceinline__ uint32_t held(uint32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}
template <uint32_t kT>
struct Seg8;

template <>
struct Seg8<FMX_TYPE_F32> {
    gm_u32x4 a, b;
    __device__ __forceinline__ void load(const uint8_t *row, uint32_t e) {
        a = *reinterpret_cast<const gm_u32x4 *>(row + 4ull * e);
        b = *reinterpret_cast<const gm_u32x4 *>(row + 4ull * e + 16);
    }
    __device__ __forceinline__ void decode(uint32_t, float (&o)[8]) const {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            o[j] = __builtin_bit_cast(float, static_cast<uint32_t>(a[j]));
            o[4 + j] = __builtin_bit_cast(float, static_cast<uint32_t>(b[j]));
        }
    }
};

template <>
struct Seg8<FMX_TYPE_Q4_0> {
    gm_u32x2 q;
    uint32_t d;
    __device__ __forceinline__ void load(const uint8_t *row, uint32_t e) {
        const uint8_t *blk = row + static_cast<uint64_t>(e / 32) * 18;
        d = *reinterpret_cast<const gm_u16 *>(blk);
        q = *reinterpret_cast<const gm_u32x2 *>(blk + 2 + (e & 8));
    }
    __device__ __forceinline__ void decode(uint32_t e, float (&o)[8]) const {
        // elements 0-15 of a block are the low nibbles, 16-31 the high ones
        const uint32_t sh = (e & 16) ? 4 : 0, w[2] = {held(q[0]), held(q[1])};
        const float df = half_bits_to_float(held(d));
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = df * (ubyte_f32((w[j >> 2] >> sh) & 0x0F0F0F0Fu, j & 3) - 8.0f);
    }
};

template <>
struct Seg8<FMX_TYPE_Q8_0> {
    gm_u32x2 q;
    uint32_t d;
    __device__ __forceinline__ void load(const uint8_t *row, uint32_t e) {
        const uint8_t *blk = row + static_cast<uint64_t>(e / 32) * 34;
        d = *reinterpret_cast<const gm_u16 *>(blk);
        q = *reinterpret_cast<const gm_u32x2 *>(blk + 2 + (e & 24));
    }
    __device__ __forceinline__ void decode(uint32_t, float (&o)[8]) const {
        const uint32_t w[2] = {held(q[0]), held(q[1])};
        const float df = half_bits_to_float(held(d));
#pragma unroll
        for (int j = 0; j < 8; ++j)
            o[j] = df * static_cast<float>(static_cast<int32_t>(w[j >> 2] << (24 - 8 * (j & 3))) >> 24);
    }
};

template <>
struct Seg8<FMX_TYPE_Q4_K> {
    gm_u32x2 q;
    gm_u32x4 h;
    __device__ __forceinline__ void load(const uint8_t *row, uint32_t e) {
        const uint8_t *blk = row + static_cast<uint64_t>(e / 256) * 144;
        h = *reinterpret_cast<const gm_u32x4 *>(blk);
        q = *reinterpret_cast<const gm_u32x2 *>(blk + 16 + 32 * ((e & 255) / 64) + (e & 31));
    }
    __device__ __forceinline__ void decode(uint32_t e, float (&o)[8]) const {
        // sub-block j = (e % 256) / 32; its 6-bit scale and min from bytes
        // j % 4 of the header's three scale dwords (quant.cpp:63-71)
        const uint32_t j = (e & 255) / 32, sh = 8 * (j & 3), dd = held(h[0]);
        const uint32_t b1 = (held(h[1]) >> sh) & 0xFFu, b2 = (held(h[2]) >> sh) & 0xFFu, b3 = (held(h[3]) >> sh) & 0xFFu;
        const uint32_t sc = j < 4 ? b1 & 63u : (b3 & 15u) | ((b1 >> 6) << 4);
        const uint32_t m = j < 4 ? b2 & 63u : (b3 >> 4) | ((b2 >> 6) << 4);
        const float d1 = half_bits_to_float(dd & 0xFFFFu) * static_cast<float>(sc);
        const float m1 = half_bits_to_float(dd >> 16) * static_cast<float>(m);
        const uint32_t nib = (j & 1) ? 4 : 0, w[2] = {held(q[0]), held(q[1])};
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = d1 * ubyte_f32((w[i >> 2] >> nib) & 0x0F0F0F0Fu, i & 3) - m1;
    }
};

template <>
struct Seg8<FMX_TYPE_Q6_K> {
    gm_u32x2 ql, qh;
    uint32_t sc, d;
    __device__ __forceinline__ void load(const uint8_t *row, uint32_t e) {
        const uint8_t *blk = row + static_cast<uint64_t>(e / 256) * 210;
        const uint32_t r = e & 255, n = r / 128, qt = (r & 127) / 32, l = r & 31;
        ql = *reinterpret_cast<const gm_u32x2 *>(blk + 64 * n + l + 32 * (qt & 1));
        qh = *reinterpret_cast<const gm_u32x2 *>(blk + 128 + 32 * n + l);
        sc = blk[192 + 8 * n + l / 16 + 2 * qt];
        d = *reinterpret_cast<const gm_u16 *>(blk + 208);
    }
    __device__ __forceinline__ void decode(uint32_t e, float (&o)[8]) const {
        const uint32_t qt = (e & 127) / 32, nib = qt >= 2 ? 4 : 0;
        const float ds = half_bits_to_float(held(d)) * static_cast<float>(static_cast<int8_t>(held(sc)));
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t w =
                ((held(ql[i]) >> nib) & 0x0F0F0F0Fu) | (((held(qh[i]) >> (2 * qt)) & 0x03030303u) << 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) o[4 * i + j] = ds * (ubyte_f32(w, j) - 32.0f);
        }
    }
};

// 32 weight rows (the result's columns) x 32 TT tokens (its rows).
// grid: (ceil(out_dim / 32), ceil(tokens / (32 TT))).
// Bound: the f32 matrix rate (two flops per weight and token at 256 per cycle
// and CU). Two workgroups per CU (52 KiB of LDS and at most 256 registers
// each at TT = 2), so that one's barrier and LDS latency run beside the
// other's MFMAs. Q8_0 [4096 x 4096] over 256 tokens: 178 us as vector FMAs
// (48 TFLOP/s), 83 us here (104 TFLOP/s; a large f32 library product reaches
// 153); over 512 tokens 351 -> 162 us; [1024 x 4096] over 8 tokens 74 -> 30
// us. On the way: MFMAs alone with one stage requested ahead 100 us, two
// ahead 95 us, the decoding dealt out between the MFMAs 88 us, held() 83 us.
template <uint32_t kT, uint32_t TT>
__global__ __launch_bounds__(kCmThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_quant_kernel(
    const uint8_t *__restrict__ w, const float *__restrict__ x, float *__restrict__ y, uint32_t tokens,
    uint32_t out_dim, uint32_t in_dim, uint64_t row_bytes) {
    constexpr uint32_t kXRows = 32 * TT, kBuf = (kXRows + kGmRows) * kGmStride;
    __shared__ __align__(16) float lds[2 * kBuf];
    static_assert(2 * kBuf >= 8192, "the chains are joined through the stage buffers");
    const uint32_t tid = threadIdx.x;
    const uint32_t o0 = blockIdx.x * kGmRows, t0 = blockIdx.y * kXRows;
    const uint32_t nc = in_dim / 8 * 8; // the chains' elements: whole groups of 8
    const uint32_t stages = (nc + kGmK - 1) / kGmK;
    // weights: row tid / 8, elements 8 (tid % 8) .. +7 of the stage
    const uint32_t wr = tid >> 3, we = 8 * (tid & 7);
    const uint8_t *wrow = w + (o0 + wr < out_dim ? o0 + wr : out_dim - 1) * row_bytes;
    // inputs: tokens tid / 16 + 16 i, elements 4 (tid % 16) .. +3
    const uint32_t xe = 4 * (tid & 15);
    const float *xrow[2 * TT];
#pragma unroll
    for (uint32_t i = 0; i < 2 * TT; ++i) {
        const uint32_t t = t0 + (tid >> 4) + 16 * i;
        xrow[i] = x + static_cast<uint64_t>(t < tokens ? t : tokens - 1) * in_dim;
    }
    // PF stages requested ahead, in PF register sets
    constexpr uint32_t PF = TT == 1 ? 4 : 2;
    Seg8<kT> seg[PF];
    gm_f32x4 xv[PF][2 * TT];
    // kFull: a stage of whole elements (all but the last one); elsewhere the
    // elements past the chains' end are not read (element 0 is, and dropped)
    auto load = [&](auto full, uint32_t p, uint32_t st) {
        constexpr bool kFull = decltype(full)::value;
        const uint32_t k0 = st * kGmK;
        seg[p].load(wrow, kFull || k0 + we < nc ? k0 + we : 0);
        const uint32_t e = kFull || k0 + xe < nc ? k0 + xe : 0;
#pragma unroll
        for (uint32_t i = 0; i < 2 * TT; ++i) xv[p][i] = *reinterpret_cast<const gm_f32x4 *>(xrow[i] + e);
    };
    auto store = [&](auto full, uint32_t p, uint32_t st) {
        constexpr bool kFull = decltype(full)::value;
        float *xs = lds + (st & 1) * kBuf, *ws = xs + kXRows * kGmStride;
        const uint32_t k0 = st * kGmK;
        float v[8];
        seg[p].decode(k0 + we, v);
        const bool win = kFull || k0 + we < nc, xin = kFull || k0 + xe < nc;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = win ? v[j] : 0.0f;
        float4 *wd = reinterpret_cast<float4 *>(ws + wr * kGmStride + we);
        wd[0] = make_float4(v[0], v[1], v[2], v[3]);
        wd[1] = make_float4(v[4], v[5], v[6], v[7]);
#pragma unroll
        for (uint32_t i = 0; i < 2 * TT; ++i)
            *reinterpret_cast<float4 *>(xs + ((tid >> 4) + 16 * i) * kGmStride + xe) =
                xin ? make_float4(xv[p][i].x, xv[p][i].y, xv[p][i].z, xv[p][i].w)
                    : make_float4(-0.0f, -0.0f, -0.0f, -0.0f);
    };
    const std::true_type full{};
    const std::false_type any{};
    ChainAcc<TT> acc;
    acc.zero();
    if (stages > 0) {
#pragma unroll
        for (uint32_t p = 0; p < PF; ++p) load(any, p, p);
        store(any, 0, 0);
        load(any, 0, PF);
        __syncthreads();
    }
    // step st: the MFMAs of stage st, stage st + 1 decoded into the other
    // buffer, stage st + 1 + PF requested. While stages up to st + 1 are
    // whole, one basic block: the decoding's vector instructions are dealt
    // out between the MFMAs, whose 64 cycles each cover about ten of them
    // (a wavefront that decodes after its MFMAs leaves the matrix unit idle
    // meanwhile).
    const uint32_t whole = nc / kGmK;
    uint32_t s0 = 0;
    for (; s0 + PF + 1 <= whole; s0 += PF) {
#pragma unroll
        for (uint32_t u = 0; u < PF; ++u) {
            const uint32_t st = s0 + u, p = (u + 1) % PF, nx = st + 1 + PF;
            const float *xs = lds + (st & 1) * kBuf;
            acc.template stage<kGmK>(xs, xs + kXRows * kGmStride);
            store(full, p, st + 1);
            load(full, p, nx < whole ? nx : whole - 1);
#pragma unroll
            for (uint32_t i = 0; i < 2 * (TT + 1); ++i) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0); // LDS reads
#pragma unroll
            for (uint32_t i = 0; i < 8 * TT; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // an MFMA
                __builtin_amdgcn_sched_group_barrier(0x002, TT == 1 ? 10 : 6, 0); // vector instructions
            }
            __syncthreads();
        }
    }
    // the last stages; `load(full)` above may have clamped the requests of
    // a partial last stage, so every set is requested again
    if (s0 > 0) {
#pragma unroll
        for (uint32_t p = 0; p < PF; ++p) load(any, (p + 1) % PF, s0 + 1 + p);
    }
    for (; s0 < stages; s0 += PF) {
#pragma unroll
        for (uint32_t u = 0; u < PF; ++u) {
            const uint32_t st = s0 + u, p = (u + 1) % PF;
            if (st >= stages) break;
            const float *xs = lds + (st & 1) * kBuf;
            acc.template stage<kGmK>(xs, xs + kXRows * kGmStride);
            store(any, p, st + 1);
            load(any, p, st + 1 + PF);
            __syncthreads();
        }
    }
    acc.finish(lds, [&](uint32_t row, uint32_t col, float total) {
        const uint32_t t = t0 + row, o = o0 + col;
        if (t >= tokens || o >= out_dim) return;
        // dot_avx2's scalar tail (F32 rows: block types are whole groups of 8)
        if constexpr (kT == FMX_TYPE_F32) {
            const uint8_t *wt = w + o * row_bytes;
            const float *xt = x + static_cast<uint64_t>(t) * in_dim;
            for (uint32_t k = nc; k < in_dim; ++k)
                total = fma_rn(__builtin_bit_cast(float, static_cast<uint32_t>(*reinterpret_cast<const gm_u32 *>(wt + 4ull * k))),
                               xt[k], total);
        }
        y[static_cast<uint64_t>(t) * out_dim + o] = total;
    });
}

template <uint32_t kT>
int launch_gemm(const void *w, const float *x, float *y, uint32_t tokens, uint32_t out_dim, uint32_t in_dim,
                uint64_t row_bytes, hipStream_t s) {
    const uint8_t *wb = static_cast<const uint8_t *>(w);
    // 64 tokens per workgroup halve the decoding per token; up to 32 tokens
    // the second half would be all padding
    if (tokens > 32)
        hipLaunchKernelGGL((gemm_quant_kernel<kT, 2>), dim3(div_up(out_dim, kGmRows), div_up(tokens, 64)),
                           dim3(kCmThreads), 0, s, wb, x, y, tokens, out_dim, in_dim, row_bytes);
    else
        hipLaunchKernelGGL((gemm_quant_kernel<kT, 1>), dim3(div_up(out_dim, kGmRows), div_up(tokens, 32)),
                           dim3(kCmThreads), 0, s, wb, x, y, tokens, out_dim, in_dim, row_bytes);
    FMX_LAUNCH_CHECK();
    return FMX_OK;
}

} // namespace
} // namespace fmx

using namespace fmx;

extern "C" int fmx_gemm_quant(uint32_t type_id, const void *weights, const float *x, float *y, uint32_t tokens,
                              uint32_t out_dim, uint32_t in_dim, void *stream) {
    if (int rc = fault_gate()) return rc;
    if (tokens == 0 || out_dim == 0 || in_dim == 0) return FMX_OK;
    if (!weights || !x || !y) return FMX_ERR_INVALID_ARGUMENT;
    uint32_t bs = 0, bb = 0;
    if (int rc = raw_geometry(type_id, &bs, &bb)) return rc;
    if (in_dim % bs) return FMX_ERR_SHAPE_MISMATCH;
    const uint64_t row_bytes = static_cast<uint64_t>(in_dim / bs) * bb;
    hipStream_t s = static_cast<hipStream_t>(stream);
    switch (type_id) {
    case FMX_TYPE_F32: return launch_gemm<FMX_TYPE_F32>(weights, x, y, tokens, out_dim, in_dim, row_bytes, s);
    case FMX_TYPE_Q4_0: return launch_gemm<FMX_TYPE_Q4_0>(weights, x, y, tokens, out_dim, in_dim, row_bytes, s);
    case FMX_TYPE_Q8_0: return launch_gemm<FMX_TYPE_Q8_0>(weights, x, y, tokens, out_dim, in_dim, row_bytes, s);
    case FMX_TYPE_Q4_K: return launch_gemm<FMX_TYPE_Q4_K>(weights, x, y, tokens, out_dim, in_dim, row_bytes, s);
    case FMX_TYPE_Q6_K: return launch_gemm<FMX_TYPE_Q6_K>(weights, x, y, tokens, out_dim, in_dim, row_bytes, s);
    }
    return FMX_ERR_UNSUPPORTED_QUANTISATION;
}
