// chain_mfma.hpp — the reference's dot_avx2 / gemv_avx2_row chains on the f32
// matrix cores.
//
// A dot of n elements in that order (kernels.cpp:147-167, 206-223) is 16
// chains, chain c a sequence of FMAs over the elements k = 16 s + c, s
// ascending; then acc_c + acc_(c+8), the 8-lane tree, and an FMA tail. The
// gfx950 f32 MFMAs add their products one FMA at a time, k ascending, each
// rounded to nearest even with denormals kept: v_mfma_f32_32x32x2_f32 with
// its two k slices set to steps s and s + 1 of chain c is two steps of that
// chain for 32 x 32 dots, bit for bit (checked on the GPU against scalar
// FMAs over normal, denormal, overflowing and mixed operands, 4 million
// outputs each). That is 256 flops per cycle and CU, twice what the vector
// unit does without packed instructions, and one operand register per 32
// rows instead of one per row.
//
// A workgroup of four wavefronts owns 32 MT rows of A x 32 rows of B (A's
// rows become the rows of the result, B's its columns); wavefront w runs the
// chains 4 w .. 4 w + 3, so that a lane's operands of its four chains are 4
// consecutive floats of a row, one 16-byte LDS read. Elements past the
// chains' end are staged as +0 in one operand and -0 in the other: the
// product is -0, and adding -0 changes no accumulator.
#pragma once

#include "fmx_internal.hpp"

namespace fmx {

typedef float fmx_f32x16 __attribute__((ext_vector_type(16)));

constexpr uint32_t kCmThreads = 256;

// Floats between staged rows of K elements: rows 4 banks apart (mod 64), so
// the 16-byte reads of 16 consecutive rows touch all 64 banks once.
template <uint32_t K>
constexpr uint32_t cm_stride() {
    static_assert(K % 64 == 0, "stages are whole multiples of 64 elements");
    return K + 4;
}

// The accumulators of one wavefront: chain 4 w + j of row block m.
template <uint32_t MT>
struct ChainAcc {
    fmx_f32x16 v[4][MT];

    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (uint32_t m = 0; m < MT; ++m)
#pragma unroll
                for (int i = 0; i < 16; ++i) v[j][m][i] = 0.0f;
    }

    // The chains' steps over one stage of K elements: `a` holds 32 MT rows,
    // `b` 32 rows (cm_stride<K>() floats apart). The operands of the next 32
    // elements are read during the MFMAs of the current ones.
    template <uint32_t K>
    __device__ __forceinline__ void stage(const float *a, const float *b) {
        const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const uint32_t at = (lane & 31) * cm_stride<K>() + 16 * (lane >> 5) + 4 * wave;
        const float *ap = a + at, *bp = b + at;
        float4 av[2][MT], bv[2];
        auto read = [&](int i, uint32_t k) {
#pragma unroll
            for (uint32_t m = 0; m < MT; ++m)
                av[i][m] = *reinterpret_cast<const float4 *>(ap + m * 32 * cm_stride<K>() + k);
            bv[i] = *reinterpret_cast<const float4 *>(bp + k);
        };
        read(0, 0);
#pragma unroll
        for (uint32_t k = 0; k < K; k += 32) {
            const int c = (k / 32) & 1;
            if (k + 32 < K) read(c ^ 1, k + 32);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float bj = j == 0 ? bv[c].x : j == 1 ? bv[c].y : j == 2 ? bv[c].z : bv[c].w;
#pragma unroll
                for (uint32_t m = 0; m < MT; ++m) {
                    const float4 q = av[c][m];
                    const float aj = j == 0 ? q.x : j == 1 ? q.y : j == 2 ? q.z : q.w;
                    v[j][m] = __builtin_amdgcn_mfma_f32_32x32x2f32(aj, bj, v[j][m], 0, 0, 0);
                }
            }
        }
    }

    // Joins the 16 chains of every dot through `ex` (LDS, 8192 floats, free
    // when every wavefront calls it) and hands each to put(row, column,
    // value), row < 32 MT, column < 32: (acc_c + acc_(c+8)) for c < 8, then
    // (s0 + s1) + (s2 + s3) with s_i = t_i + t_(i+4). Each wavefront joins a
    // quarter of the result's registers; consecutive lanes get consecutive
    // columns.
    template <class Put>
    __device__ __forceinline__ void finish(float *ex, Put put) {
        const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
        for (uint32_t m = 0; m < MT; ++m) {
#pragma unroll
            for (uint32_t half = 0; half < 2; ++half) {
                __syncthreads();
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j)
#pragma unroll
                    for (uint32_t r = 0; r < 8; ++r) ex[((4 * wave + j) * 8 + r) * 64 + lane] = v[j][m][8 * half + r];
                __syncthreads();
#pragma unroll
                for (uint32_t u = 0; u < 2; ++u) {
                    const uint32_t r = 2 * wave + u;
                    float t[8];
#pragma unroll
                    for (uint32_t c = 0; c < 8; ++c)
                        t[c] = ex[(c * 8 + r) * 64 + lane] + ex[((c + 8) * 8 + r) * 64 + lane];
                    const float total = ((t[0] + t[4]) + (t[1] + t[5])) + ((t[2] + t[6]) + (t[3] + t[7]));
                    const uint32_t rr = 8 * half + r;
                    put(32 * m + 8 * (rr >> 2) + 4 * (lane >> 5) + (rr & 3), lane & 31, total);
                }
            }
        }
    }
};

} // namespace fmx
