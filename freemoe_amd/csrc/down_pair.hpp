// down_pair.hpp — the down projection of one decode token on 16 lanes per
// row (Q4_0 and Q4_K down matrices); included by moe.hip (Q4_0) and
// down_pair_q4k.hip (Q4_K), each instantiating its own block type.
#pragma once

#include "moe.hpp"
#include "pair.hpp"

#include <hip/hip_ext.h>

namespace fmx {

namespace {

// Prefetch depth (chunks in flight per row) and the dynamic LDS a launch may
// request (a gfx950 workgroup holds 160 KiB, 1 KiB left for static LDS).
constexpr int kPairPF = 7;
constexpr size_t kPairMaxLds = 159 * 1024;

// Down rows as down_kernel, on twice the lanes: 16 per row slot (pair.hpp), 512
// threads, two wavefronts per SIMD (Q4_0 and Q4_K down matrices); the row's
// result is down_kernel's bit for bit. The ranks' activations, one after
// another in memory, fill the LDS as one tile (the host checks that they fit)
// from one batch of requests: kB quads per thread hold 8192 or 32768 of them,
// the first for the many small ranks of a fine-grained layer, whose kernel is
// a chain of latencies (Q4_K, top-8 of 768: 20.7 us with the ranks past the
// second staged one by one, 12.2 us).
constexpr uint32_t kPairThreads = 512;

template <class P, int PF, int kB>
__global__ __launch_bounds__(kPairThreads) __attribute__((amdgpu_waves_per_eu(2, 2), aligned(4096))) void down_pair_kernel(
    ExpertArgs a, const float *__restrict__ x, const float *__restrict__ act, const uint32_t *__restrict__ ids,
    const float *__restrict__ w, float *__restrict__ out, uint32_t *__restrict__ status) {
    using T = typename P::T;
    extern __shared__ __align__(16) float lds[];
    __shared__ float dres[kPairThreads / 16];
    const uint32_t tid = threadIdx.x, l = tid & 7, hf = (tid >> 3) & 1, slot = tid >> 4;
    const uint32_t K = a.top_k, H = a.hidden;
    const uint32_t jpw = (kPairThreads / 16) / K;
    const uint32_t rank = slot / jpw < K ? slot / jpw : K - 1;
    const uint32_t j = blockIdx.x * jpw + slot % jpw;
    const uint32_t jr = j < H ? j : H - 1;
    uint32_t e = ids[rank];
    const bool bad = e >= a.experts;
    if (bad) {
        if ((tid & 15) == 0) atomicOr(status, STATUS_BAD_EXPERT);
        e = 0;
    }
    // quants of lane l's slice (its half) and the chunk's scales / header
    const typename T::Row rw = T::row(static_cast<const uint8_t *>(a.down[e]), a.dn.scale_bytes, a.dn.blocks_padded,
                                      a.dn.chunks, jr, l);
    const uint8_t *qp = rw.quants + 8 * hf, *sp = P::scales(rw);
    const uint32_t blocks = a.dn.blocks, c_end = blocks / T::kPerChunk;
    // the activations requested first (staging waits for its loads in issue
    // order), then the first weight chunks, then the staging
    XBatch<kB> xb;
    load_batch<T>(xb, act, 0, K * blocks * T::kBlock, tid, kPairThreads);
    PairChunk buf[PF + 1];
    pair_prime<P, PF>(qp, sp, c_end, buf);
    T::template stage<kB, true>(act, 0, K * blocks, lds, tid, kPairThreads, xb);
    __syncthreads();
    const float t = pair_stream<P, PF>(qp, sp, c_end, P::x_of(lds, K * blocks, rank * blocks, l), l, hf, buf);
    const float v = P::finish(t);
    if ((tid & 15) == 0) dres[slot] = bad ? 0.0f : v;
    __syncthreads();
    if (tid < jpw) {
        const uint32_t jo = blockIdx.x * jpw + tid;
        if (jo < H) {
            float ffn = 0.0f;
            for (uint32_t r = 0; r < K; ++r) ffn = ffn + w[r] * dres[r * jpw + tid];
            out[jo] = x[jo] + ffn;
        }
    }
}

// The 16-lane down kernel (block type P::T) serves a layer when every rank's
// activations fit the LDS as one tile and the rows are whole chunks.
template <class P>
bool pair_down_fits(const ExpertArgs &a) {
    using T = typename P::T;
    return a.type_dn == T::kType && a.top_k <= kPairThreads / 16 && a.dn.blocks % T::kPerChunk == 0 &&
           static_cast<size_t>(a.dn.blocks) * T::kLdsFloatsPerBlock * sizeof(float) * a.top_k <= kPairMaxLds;
}

template <class P>
int launch_down_pair(const ExpertArgs &a, const float *x, const float *act, const uint32_t *ids, const float *w,
                     float *out, uint32_t *status, hipStream_t s, const hipEvent_t *kev) {
    auto dn = a.top_k * a.ffn <= 4 * 4 * kPairThreads ? down_pair_kernel<P, kPairPF, 4>
                                                      : down_pair_kernel<P, kPairPF, 16>;
    const size_t lds = static_cast<size_t>(a.dn.blocks) * P::T::kLdsFloatsPerBlock * sizeof(float) * a.top_k;
    if (int rc = allow_lds(reinterpret_cast<const void *>(dn), lds)) return rc;
    const dim3 grid(div_up(a.hidden, (kPairThreads / 16) / a.top_k));
    if (kev)
        hipExtLaunchKernelGGL(dn, grid, dim3(kPairThreads), lds, s, kev[0], kev[1], 0, a, x, act, ids, w, out, status);
    else
        hipLaunchKernelGGL(dn, grid, dim3(kPairThreads), lds, s, a, x, act, ids, w, out, status);
    FMX_LAUNCH_CHECK();
    return FMX_OK;
}

} // namespace

} // namespace fmx
