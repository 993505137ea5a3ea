// matvec.hip — y = W x for one matrix (Backend::matvec / gemv_quant).
//
// Block-type rows use the lane chains of chains.hpp (Q4_0, Q8_0, Q4_K: the
// reference's dedicated AVX2 row dots); Q6_K rows, which the reference runs
// through row_dot_fused_scalar (kernels.cpp:574-590: each block decoded,
// dotted by dot_avx2, the block's dot added to the row total), use that order
// on quads of lanes, a block each; F32 rows use the
// reference's gemv_avx2_row order (kernels.cpp:147-167): per row 16 chains
// (chain c takes k = c mod 16; chains 0..7 are acc0, 8..15 acc1), an 8-element
// tail into acc0, lane-wise acc0 + acc1, the 8-lane tree sum, then a scalar
// FMA tail over the last in_dim mod 8 elements.
#include "matvec.hpp"
#include "pair.hpp"

namespace fmx {

namespace {

constexpr uint32_t kThreads = 256;              // 4 wavefronts
constexpr uint32_t kLdsBudgetFloats = 8 * 1024; // 32 KiB of x per tile
constexpr size_t kMatvecMaxLds = 128 * 1024;     // the pair kernel's x
constexpr size_t kQ6MaxLds = 159 * 1024;         // the Q6_K quad kernel's x and dots
constexpr uint32_t kQ6Quads = 131072;            // eight wavefronts per SIMD

template <class T, int NR>
__global__ __launch_bounds__(kThreads) void matvec_kernel(
    const uint8_t *__restrict__ packed, const float *__restrict__ x, float *__restrict__ y,
    uint32_t rows, uint32_t blocks, uint32_t blocks_padded, uint32_t chunks, uint64_t scale_bytes,
    uint32_t tile_blocks) {
    extern __shared__ __align__(16) float lds[];
    const uint32_t tid = threadIdx.x;
    const uint32_t l = tid & 7;
    const uint32_t slot = tid >> 3; // 0..31
    const uint32_t r0 = (blockIdx.x * (kThreads / 8) + slot) * NR;
    typename T::Row rw[NR];
    float t[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
        const uint32_t r = r0 + i < rows ? r0 + i : rows - 1; // clamp: loads stay in bounds
        rw[i] = T::row(packed, scale_bytes, blocks_padded, chunks, r, l);
        t[i] = 0.0f;
    }
    for (uint32_t tb = 0; tb < blocks; tb += tile_blocks) {
        const uint32_t nb = blocks - tb < tile_blocks ? blocks - tb : tile_blocks;
        __syncthreads();
        T::stage(x, tb, nb, lds, tid, kThreads);
        __syncthreads();
        const uint32_t c0 = tb / T::kPerChunk;
        const uint32_t c1 = (tb + nb + T::kPerChunk - 1) / T::kPerChunk;
        run_chunks_pf<T, NR, 2>(rw, c0, c1, blocks, tb, nb, lds, l, t);
    }
#pragma unroll
    for (int i = 0; i < NR; ++i) {
        const float v = T::finish(t[i]);
        if (l == 0 && r0 + i < rows) y[r0 + i] = v;
    }
}

// Two 8-lane groups per row (pair.hpp), 16 rows per workgroup, x as one LDS
// tile, the rows' first PF chunks requested before it is staged.
template <class P, int PF>
__global__ __launch_bounds__(kThreads) void matvec_pair_kernel(
    const uint8_t *__restrict__ packed, const float *__restrict__ x, float *__restrict__ y, uint32_t rows,
    uint32_t blocks, uint32_t chunks, uint64_t scale_bytes) {
    using T = typename P::T;
    extern __shared__ __align__(16) float lds[];
    const uint32_t tid = threadIdx.x, l = tid & 7, hf = (tid >> 3) & 1;
    const uint32_t r = blockIdx.x * (kThreads / 16) + (tid >> 4);
    const typename T::Row rw = T::row(packed, scale_bytes, blocks, chunks, r < rows ? r : rows - 1, l);
    const uint8_t *qp = rw.quants + 8 * hf, *sp = P::scales(rw);
    XBatch<4> xb;
    load_batch<T>(xb, x, 0, blocks * T::kBlock, tid, kThreads);
    PairChunk buf[PF + 1];
    pair_prime<P, PF>(qp, sp, chunks, buf);
    T::template stage<4, true>(x, 0, blocks, lds, tid, kThreads, xb);
    __syncthreads();
    const float v = P::finish(pair_stream<P, PF>(qp, sp, chunks, P::x_of(lds, blocks, 0, l), l, hf, buf));
    if ((tid & 15) == 0 && r < rows) y[r] = v;
}

// F32: 16 lanes per row (4 row slots per wavefront, 16 per workgroup).
// kXs: x staged in LDS first (n floats), so each input is read from memory
// once per workgroup instead of once per row; the groups of a wavefront read
// the same elements at once.
template <bool kXs>
__global__ __launch_bounds__(kThreads) void matvec_f32_kernel(const float *__restrict__ w,
                                                              const float *__restrict__ x,
                                                              float *__restrict__ y,
                                                              uint32_t rows, uint32_t n) {
    extern __shared__ __align__(16) float xs_f32[];
    const uint32_t tid = threadIdx.x;
    const uint32_t c = tid & 15;
    const float *xr = x;
    if constexpr (kXs) {
        if ((reinterpret_cast<uintptr_t>(x) & 15u) == 0 && n % 4 == 0) {
            const float4 *x4 = reinterpret_cast<const float4 *>(x);
            for (uint32_t q = tid; q < n / 4; q += kThreads) reinterpret_cast<float4 *>(xs_f32)[q] = x4[q];
        } else {
            for (uint32_t q = tid; q < n; q += kThreads) xs_f32[q] = x[q];
        }
        __syncthreads();
        xr = xs_f32;
    }
    const uint32_t r = blockIdx.x * (kThreads / 16) + (tid >> 4);
    const uint32_t rr = r < rows ? r : rows - 1;
    const float *row = w + static_cast<uint64_t>(rr) * n;
    const float total = f32_row_chains<true>(row, xr, n, c);
    if (c == 0 && r < rows) y[r] = total;
}

// Q6_K: 16 lanes per row over raw blocks (q6_k_row_chains).
__global__ __launch_bounds__(kThreads) void matvec_q6_k_kernel(const uint8_t *__restrict__ w,
                                                               const float *__restrict__ x,
                                                               float *__restrict__ y, uint32_t rows,
                                                               uint32_t blocks) {
    const uint32_t tid = threadIdx.x, c = tid & 15;
    const uint32_t r = blockIdx.x * (kThreads / 16) + (tid >> 4);
    const uint32_t rr = r < rows ? r : rows - 1;
    const float total = q6_k_row_chains(w + static_cast<uint64_t>(rr) * blocks * 210, x, blocks, c);
    if (c == 0 && r < rows) y[r] = total;
}

// Q6_K, four 16-lane groups per row, group g taking blocks g, g + 4, ..., x from
// memory; the block dots meet in LDS (4 rows x blocks) and one lane adds them in
// block order from 0, as q6_k_row_chains does.
__global__ __launch_bounds__(kThreads) void matvec_q6_k_split_kernel(const uint8_t *__restrict__ w,
                                                                     const float *__restrict__ x,
                                                                     float *__restrict__ y, uint32_t rows,
                                                                     uint32_t blocks) {
    extern __shared__ __align__(16) float q6_lds[];
    constexpr uint32_t kRows = kThreads / 64;
    const uint32_t tid = threadIdx.x, lr = tid >> 6, r0 = blockIdx.x * kRows;
    const uint8_t *row = w + static_cast<uint64_t>(r0 + lr < rows ? r0 + lr : rows - 1) * blocks * 210;
    q6_k_block_dots(row, x, blocks, (tid >> 4) & 3, 4, tid & 15, q6_lds + lr * blocks);
    __syncthreads();
    if (tid < kRows && r0 + tid < rows) y[r0 + tid] = q6_sum_dots(q6_lds + tid * blocks, blocks);
}

// Q6_K with x in LDS (block b at xs + b * kQ6XStride): a quad of lanes works on
// one block at a time (Q6Quad), G quads per row, quad g taking blocks g,
// g + G, ... (each block's dot is independent); the block dots meet in LDS and
// one lane adds them in block order from 0, as q6_k_row_chains does.
// LDS: NT / 4 / G rows x blocks dots, then x.
template <uint32_t NT, uint32_t G>
__global__ __launch_bounds__(NT) void matvec_q6_k_quad_kernel(const uint8_t *__restrict__ w,
                                                                    const float *__restrict__ x, float *__restrict__ y,
                                                                    uint32_t rows, uint32_t blocks) {
    extern __shared__ __align__(16) float q6_lds[];
    constexpr uint32_t kRows = NT / 4 / G;
    float *dots = q6_lds, *xs = q6_lds + q6_dots_floats(kRows, blocks);
    const uint32_t tid = threadIdx.x, i = tid & 3, quad = tid >> 2;
    const uint32_t lr = quad / G, part = quad % G;
    const uint32_t r = blockIdx.x * kRows + lr;
    const uint8_t *row = w + static_cast<uint64_t>(r < rows ? r : rows - 1) * blocks * 210;
    Q6Quad first;
    first.load(row + (part < blocks ? part : 0) * 210, i);
    q6_stage_x(x, blocks * 256, xs, tid, NT);
    __syncthreads();
    q6_quad_block_dots(first, row, xs, blocks, part, G, i, dots + lr * blocks);
    __syncthreads();
    if (tid < kRows && blockIdx.x * kRows + tid < rows) y[blockIdx.x * kRows + tid] = q6_sum_dots(dots + tid * blocks, blocks);
}

template <uint32_t NT, uint32_t G>
int launch_q6_k_quad(const void *w, const float *x, float *y, uint32_t rows, uint32_t blocks, hipStream_t s, bool *done) {
    constexpr uint32_t kRows = NT / 4 / G;
    const size_t lds = (q6_dots_floats(kRows, blocks) + static_cast<size_t>(blocks) * kQ6XStride) * sizeof(float);
    *done = lds <= kQ6MaxLds;
    if (!*done) return FMX_OK;
    auto k = matvec_q6_k_quad_kernel<NT, G>;
    if (int rc = allow_lds(reinterpret_cast<const void *>(k), lds)) return rc;
    hipLaunchKernelGGL(k, dim3(div_up(rows, kRows)), dim3(NT), lds, s, static_cast<const uint8_t *>(w), x, y,
                       rows, blocks);
    FMX_LAUNCH_CHECK();
    return FMX_OK;
}

// The quad kernel's layout for a Q6_K matrix (*done: whether x and the dots fit
// the LDS). Every workgroup stages x, so long rows (32 blocks and more, where
// few workgroups of 256 threads share a CU's LDS) take larger ones; past 80
// blocks one fills a CU, and its threads and quads are such that the device's
// 256 workgroups hold the rows. [4096 x 8192] 8.5 us on 512 threads and 16 quads
// a row, [6144 x 14336] 20.7 (1024 threads 27.5, x not staged 24.4), [16384 x
// 14336] on 8 quads 40.9 (256 threads 50.3); [5120 x 27648] 1024 threads and 8
// quads 40 (x not staged 39, one lane group a row 73), [4096 x 25088] 23 (30, 56),
// [2048 x 24576] 512 threads and 16 quads 13.2 (18.9).
// Shorter rows: with few rows the chain over a row's blocks bounds, as many quads
// as it has blocks ([1024 x 1536] eight 3.5, four 4.2; up to eight blocks as long
// as the rows leave room, [12288 x 1280] eight 6.4, two 6.8); with more, the
// device is full and quads without a block are lost: the most quads that leave
// at most a fifth idle ([8192 x 5120] 16, 8, 4 quads 12.9, 11.3, 10.4; [4096 x 2560] 5.4,
// 5.6, 5.3; [16384 x 2560] eight 13.1, four 11.1).
int launch_q6_k_quads(const void *w, const float *x, float *y, uint32_t rows, uint32_t blocks, hipStream_t s, bool *done) {
    const uint32_t want = kQ6Quads / rows; // quads per row that fill the device
    if (blocks > 80 && rows > 1024) {
        if (rows <= 2048) return launch_q6_k_quad<512, 16>(w, x, y, rows, blocks, s, done);
        if (rows <= 4096) return launch_q6_k_quad<1024, 16>(w, x, y, rows, blocks, s, done);
        if (rows <= 8192) return launch_q6_k_quad<1024, 8>(w, x, y, rows, blocks, s, done);
        return launch_q6_k_quad<512, 8>(w, x, y, rows, blocks, s, done);
    }
    if (blocks >= 32 && rows >= 4096 && want >= 8)
        return want >= 16 ? launch_q6_k_quad<512, 16>(w, x, y, rows, blocks, s, done)
                          : launch_q6_k_quad<512, 8>(w, x, y, rows, blocks, s, done);
    uint32_t g = 16;
    if (blocks <= 8 ? want > 8 : blocks <= 16 ? want >= 32 : want >= 128)
        while (g / 2 >= blocks) g /= 2;
    else
        while (g > 1 && (g > want || 4 * div_up(blocks, g) * g > 5 * blocks)) g /= 2;
    switch (g) {
    case 16: return launch_q6_k_quad<256, 16>(w, x, y, rows, blocks, s, done);
    case 8: return launch_q6_k_quad<256, 8>(w, x, y, rows, blocks, s, done);
    case 4: return launch_q6_k_quad<256, 4>(w, x, y, rows, blocks, s, done);
    case 2: return launch_q6_k_quad<256, 2>(w, x, y, rows, blocks, s, done);
    }
    return launch_q6_k_quad<256, 1>(w, x, y, rows, blocks, s, done);
}

// Q6_K: the quads, but x staged and the dots joined cost more than they save
// where a row is over at once (GPU time): up to three blocks on 16 lanes
// ([4096 x 512] 2.6 us, quads 3.4; [12288 x 768] 4.5, 4.5), and with few rows
// where the quads' second round is mostly idle or their one round long, on four
// groups of 16 lanes ([1024 x 2048] 2.9, quads 3.5; x 3072 3.4, 3.6; x 5120 4.4,
// 4.7; but x 4096 3.8, 3.6). x past the LDS: four groups below 8192 rows
// ([1024 x 28672] 15 us, one group 49), one from there ([8192 x 28672] 74, two
// 138).
int launch_matvec_q6_k(const void *w, const float *x, float *y, uint32_t rows, uint32_t blocks, hipStream_t s) {
    const uint8_t *wb = static_cast<const uint8_t *>(w);
    auto split = [&]() -> int {
        hipLaunchKernelGGL(matvec_q6_k_split_kernel, dim3(div_up(rows, kThreads / 64)), dim3(kThreads),
                           kThreads / 64 * blocks * sizeof(float), s, wb, x, y, rows, blocks);
        FMX_LAUNCH_CHECK();
        return FMX_OK;
    };
    const bool one = blocks <= 3 && rows <= (blocks == 1 ? 32768 : 12288);
    if (!one) {
        if (rows <= 1024 && ((blocks >= 8 && blocks <= 12) || (blocks >= 17 && blocks <= 20))) return split();
        bool done;
        if (int rc = launch_q6_k_quads(w, x, y, rows, blocks, s, &done)) return rc;
        if (done) return FMX_OK;
        if (rows < 8192 && blocks <= 4096) return split(); // (64 KiB of dots)
    }
    hipLaunchKernelGGL(matvec_q6_k_kernel, dim3(div_up(rows, kThreads / 16)), dim3(kThreads), 0, s, wb, x, y, rows,
                       blocks);
    FMX_LAUNCH_CHECK();
    return FMX_OK;
}

template <class T, int NR>
int launch_matvec(const PackedGeometry &g, const void *packed, const float *x, float *y,
                  hipStream_t s) {
    const uint32_t tb = tile_blocks_for<T>(g.blocks, kLdsBudgetFloats);
    const size_t lds = static_cast<size_t>(tb) * T::kLdsFloatsPerBlock * sizeof(float);
    const uint32_t rows_per_wg = (kThreads / 8) * NR;
    hipLaunchKernelGGL((matvec_kernel<T, NR>), dim3(div_up(g.rows, rows_per_wg)), dim3(kThreads),
                       lds, s, static_cast<const uint8_t *>(packed), x, y, g.rows, g.blocks,
                       g.blocks_padded, g.chunks, g.scale_bytes, tb);
    FMX_LAUNCH_CHECK();
    return FMX_OK;
}

// Rows up to which the pair kernel serves a type: its twice as many wavefronts
// with seven chunks each in flight are for matrices whose rows leave the device
// short of them. [4096 x 4096] matvec_kernel -> pair: Q4_0 14.2 -> 7.2, Q8_0
// 18.3 -> 7.2, Q4_K 11.8 -> 8.5 us; [4096 x 14336] 44.9 -> 13.5, 58.2 -> 18.6,
// 34.5 -> 20.9. With more rows its 17% more instructions per block cost more,
// and sooner the shorter the rows, whose chains are short anyway (GPU time):
// Q4_0 [16384 x 4096] 14.5 -> 11.3, [32000 x 4096] 18.9 -> 19.5, [16384 x 512]
// 4.0 -> 4.2, [8192 x 256] 0.93 of it and [10240 x 256] 1.05; Q8_0 [32768 x 4096]
// 29.5 -> 26.9 but [32768 x 2048] 15.4 -> 16.8 and x 512 5.5 -> 7.1; Q4_K, the
// most per block, [4096 x 2048] 6.7 -> 5.1, [8192 x 2048] 7.2 -> 7.7, x 8192 21.5
// -> 19.8. (15 chunks in flight: the same up to 4096 rows, slower above.)
uint32_t pair_rows(uint32_t type_id, uint32_t cols) {
    if (type_id == FMX_TYPE_Q4_K) return cols >= 8192 ? 8192 : 4096;
    if (cols < 1024) return cols < 512 ? 8192 : 12288;
    if (type_id == FMX_TYPE_Q4_0 || cols < 2048) return 16384;
    return cols < 4096 ? 24576 : 32768;
}

template <class P, int NR>
int launch_matvec_quant(const PackedGeometry &g, const void *packed, const float *x, float *y, hipStream_t s) {
    using T = typename P::T;
    const size_t lds = static_cast<size_t>(g.blocks) * T::kLdsFloatsPerBlock * sizeof(float);
    if (g.rows > pair_rows(T::kType, g.blocks * T::kBlock) || g.blocks % T::kPerChunk != 0 || lds > kMatvecMaxLds)
        return launch_matvec<T, NR>(g, packed, x, y, s);
    auto k = matvec_pair_kernel<P, 7>;
    if (int rc = allow_lds(reinterpret_cast<const void *>(k), lds)) return rc;
    hipLaunchKernelGGL(k, dim3(div_up(g.rows, kThreads / 16)), dim3(kThreads), lds, s,
                       static_cast<const uint8_t *>(packed), x, y, g.rows, g.blocks, g.chunks, g.scale_bytes);
    FMX_LAUNCH_CHECK();
    return FMX_OK;
}

} // namespace

} // namespace fmx

using namespace fmx;

extern "C" int fmx_matvec(uint32_t type_id, const void *packed, const float *x, float *y,
                          uint32_t out_dim, uint32_t in_dim, void *stream) {
    if (int rc = fault_gate()) return rc;
    if (out_dim == 0 || in_dim == 0) return FMX_OK;
    PackedGeometry g;
    if (int rc = packed_geometry(type_id, out_dim, in_dim, &g)) return rc;
    if (!packed || !x || !y) return FMX_ERR_INVALID_ARGUMENT;
    // block-type kernels stage x with 16-byte loads
    if (type_id != FMX_TYPE_F32 && (reinterpret_cast<uintptr_t>(x) & 15u)) return FMX_ERR_INVALID_ARGUMENT;
    // Q6_K blocks: scales and d are read as 2-byte words
    if (type_id == FMX_TYPE_Q6_K && (reinterpret_cast<uintptr_t>(packed) & 1u)) return FMX_ERR_INVALID_ARGUMENT;
    hipStream_t s = static_cast<hipStream_t>(stream);
    switch (type_id) {
    case FMX_TYPE_F32:
        if (in_dim <= 16384)
            hipLaunchKernelGGL(matvec_f32_kernel<true>, dim3(div_up(out_dim, kThreads / 16)), dim3(kThreads),
                               static_cast<size_t>(in_dim) * sizeof(float), s, static_cast<const float *>(packed), x, y,
                               out_dim, in_dim);
        else
            hipLaunchKernelGGL(matvec_f32_kernel<false>, dim3(div_up(out_dim, kThreads / 16)), dim3(kThreads), 0, s,
                               static_cast<const float *>(packed), x, y, out_dim, in_dim);
        FMX_LAUNCH_CHECK();
        return FMX_OK;
    case FMX_TYPE_Q4_0: return launch_matvec_quant<PairQ40, 2>(g, packed, x, y, s);
    case FMX_TYPE_Q8_0: return launch_matvec_quant<PairQ80, 2>(g, packed, x, y, s);
    case FMX_TYPE_Q4_K: return launch_matvec_quant<PairQ4K, 1>(g, packed, x, y, s);
    case FMX_TYPE_Q6_K: return launch_matvec_q6_k(packed, x, y, out_dim, g.blocks, s);
    }
    return FMX_ERR_UNSUPPORTED_QUANTISATION;
}
