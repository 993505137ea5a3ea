// pair.hpp — row dots on 16 lanes per row: two 8-lane groups share a row's
// chunks (Q4_0, Q8_0, Q4_K), for the decode down kernels and the
// matrix-vector products.
//
// A row's sum is a sequence of independent per-block values folded into a
// chain in block order: Q4_0's lane chains t_l = fma(c_b, d_b, t_l) with c_b =
// (lo + hi) - 8 sum x, Q8_0's with c_b the lane's sum of products, Q4_K's
// running total t = t + (part_lo + part_hi) per 32-element group pair. Lane
// l < 8 of a slot computes the values of the first half of each chunk from its
// half of lane l's 16-byte slice, lane l + 8 those of the second half from the
// other, a DPP rotation of the 16-lane row by 8 hands the second half's values
// to lane l, and lane l folds them all in the reference's order.
#pragma once

#include "chains.hpp"

namespace fmx {

namespace {

// Lane (i + 8) mod 16's value within each row of 16 lanes (DPP row_ror:8).
__device__ __forceinline__ float row_swap8(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x128, 0xF, 0xF, false));
}

struct PairChunk {
    uint2 q; // dwords 2 hf, 2 hf + 1 of the lane's slice
    uint4 s; // the chunk's block scales (Q4_0; Q8_0 in two dwords) or super-block header (Q4_K)
};

// Q4_0: a chunk is 8 blocks; lane half hf takes blocks 4 hf .. 4 hf + 3.
struct PairQ40 {
    using T = Q40;
    static constexpr uint32_t kScaleBytes = 16; // of a chunk
    __device__ static const uint8_t *scales(const T::Row &w) { return w.scales; }
    __device__ static uint4 load_scales(const uint8_t *p) { return ld16(p); }
    static constexpr int kNV = 4;
    // this lane's quads and sums of the tile of nb_tile blocks from its block b
    // on (block stride 8, chunk stride 64)
    struct X {
        const float4 *xs4;
        const float *s8;
    };
    __device__ static X x_of(const float *tile, uint32_t nb_tile, uint32_t b, uint32_t l) {
        return X{reinterpret_cast<const float4 *>(tile) + b * 8 + l, tile + nb_tile * 32 + b * 8 + l};
    }
    // The lane's LDS operands of one chunk: blocks 4 hf + q, q < 4.
    struct XC {
        float4 xv[4];
        float s8[4];
    };
    __device__ static void read_x(const X &xt, uint32_t ch, uint32_t /*l*/, uint32_t hf, XC &o) {
        const float4 *xs4 = xt.xs4 + ch * 64;
        const float *s8 = xt.s8 + ch * 64;
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
            o.xv[q] = xs4[(4 * hf + q) * 8];
            o.s8[q] = s8[(4 * hf + q) * 8];
        }
    }
    // c of blocks 4 hf + q, q < 4, of the chunk whose operands `xc` holds.
    __device__ static void values(const PairChunk &k, const XC &xc, uint32_t /*hf*/, float (&c)[kNV]) {
#pragma unroll
        for (uint32_t jj = 0; jj < 2; ++jj) {
            const uint32_t qw = jj ? k.q.y : k.q.x;
            const uint32_t lo4 = qw & 0x0F0F0F0Fu, hi4 = (qw >> 4) & 0x0F0F0F0Fu;
#pragma unroll
            for (uint32_t h = 0; h < 2; ++h) {
                const uint32_t q = 2 * jj + h;
                const float4 xv = xc.xv[q];
                const float2 lq = h ? nibble_pair<true>(lo4) : nibble_pair<false>(lo4);
                const float2 hq = h ? nibble_pair<true>(hi4) : nibble_pair<false>(hi4);
                const float lo = fma_rn(lq.x, xv.x, lq.y * xv.y);
                const float hi = fma_rn(hq.x, xv.z, hq.y * xv.w);
                c[q] = (lo + hi) - xc.s8[q];
            }
        }
    }
    // t = fma(c_b, d_b, t) for blocks 0-7: own values, then the partner's.
    __device__ static float chain(const PairChunk &k, const float (&c)[kNV], float t) {
        float r[kNV];
#pragma unroll
        for (int q = 0; q < kNV; ++q) r[q] = row_swap8(c[q]);
        const uint32_t sw[4] = {k.s.x, k.s.y, k.s.z, k.s.w};
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const float cb = b < 4 ? c[b] : r[b - 4];
            const float d = half_bits_to_float((b & 1) ? (sw[b >> 1] >> 16) : (sw[b >> 1] & 0xFFFFu));
            t = fma_rn(cb, d, t);
        }
        return t;
    }
    __device__ static float finish(float t) { return hsum8_lanes(t); }
};

// Q8_0: a chunk is 4 blocks; lane half hf takes blocks 2 hf and 2 hf + 1.
struct PairQ80 {
    using T = Q80;
    static constexpr uint32_t kScaleBytes = 8;
    __device__ static const uint8_t *scales(const T::Row &w) { return w.scales; }
    __device__ static uint4 load_scales(const uint8_t *p) {
        const uint2 s = ld8(p);
        return make_uint4(s.x, s.y, 0, 0);
    }
    static constexpr int kNV = 2;
    struct X {
        const float4 *xs4;
    };
    __device__ static X x_of(const float *tile, uint32_t /*nb_tile*/, uint32_t b, uint32_t l) {
        return X{reinterpret_cast<const float4 *>(tile) + b * 8 + l};
    }
    struct XC {
        float4 xv[2];
    };
    __device__ static void read_x(const X &xt, uint32_t ch, uint32_t /*l*/, uint32_t hf, XC &o) {
#pragma unroll
        for (uint32_t q = 0; q < 2; ++q) o.xv[q] = xt.xs4[ch * 32 + (2 * hf + q) * 8];
    }
    // Q80::step's sum over the lane's four elements of each block.
    __device__ static void values(const PairChunk &k, const XC &xc, uint32_t /*hf*/, float (&c)[kNV]) {
#pragma unroll
        for (uint32_t q = 0; q < 2; ++q) {
            const uint32_t w = q ? k.q.y : k.q.x;
            float acc = fma_rn(Q80::sbyte(w, 0), xc.xv[q].x, 0.0f);
            acc = fma_rn(Q80::sbyte(w, 1), xc.xv[q].y, acc);
            acc = fma_rn(Q80::sbyte(w, 2), xc.xv[q].z, acc);
            c[q] = fma_rn(Q80::sbyte(w, 3), xc.xv[q].w, acc);
        }
    }
    // t = fma(c_b, d_b, t) for blocks 0-3: own values, then the partner's.
    __device__ static float chain(const PairChunk &k, const float (&c)[kNV], float t) {
        const float r0 = row_swap8(c[0]), r1 = row_swap8(c[1]);
        t = fma_rn(c[0], half_bits_to_float(k.s.x & 0xFFFFu), t);
        t = fma_rn(c[1], half_bits_to_float(k.s.x >> 16), t);
        t = fma_rn(r0, half_bits_to_float(k.s.y & 0xFFFFu), t);
        return fma_rn(r1, half_bits_to_float(k.s.y >> 16), t);
    }
    __device__ static float finish(float t) { return hsum8_lanes(t); }
};

// Q4_K: a chunk is one super-block of four 64-element group pairs; lane half
// hf takes groups 2 hf and 2 hf + 1, each reduced over its 8 lanes by the
// reference's lane tree (as Q4K::step).
struct PairQ4K {
    using T = Q4K;
    static constexpr uint32_t kScaleBytes = 16; // of a chunk
    __device__ static const uint8_t *scales(const T::Row &w) { return w.header; }
    __device__ static uint4 load_scales(const uint8_t *p) { return ld16(p); }
    static constexpr int kNV = 2;
    struct X {
        const float4 *xs;
        const float *sums;
    };
    __device__ static X x_of(const float *tile, uint32_t nb_tile, uint32_t b, uint32_t) {
        return X{reinterpret_cast<const float4 *>(tile) + b * 64, tile + nb_tile * 256 + b * 8};
    }
    // 6-bit scale / min of sub-block j = 4 hf + i (k4_scale_min, quant.cpp:63-71)
    // with i a compile-time constant and hf per lane: both forms from the
    // header's dwords 1-3, then a select.
    template <uint32_t i>
    __device__ static void scale_min(const uint4 &h, uint32_t hf, uint32_t &sc, uint32_t &m) {
        const uint32_t b1 = (h.y >> (8 * i)) & 0xFFu, b2 = (h.z >> (8 * i)) & 0xFFu, b3 = (h.w >> (8 * i)) & 0xFFu;
        sc = hf ? ((b3 & 0x0Fu) | ((b1 >> 6) << 4)) : (b1 & 63u);
        m = hf ? ((b3 >> 4) | ((b2 >> 6) << 4)) : (b2 & 63u);
    }
    // The lane's LDS operands of one super-block: groups 2 hf and 2 hf + 1.
    struct XC {
        float4 xl[2], xh[2];
        float sum_lo[2], sum_hi[2];
    };
    __device__ static void read_x(const X &xt, uint32_t ch, uint32_t l, uint32_t hf, XC &o) {
#pragma unroll
        for (uint32_t gg = 0; gg < 2; ++gg) {
            const uint32_t g = 2 * hf + gg;
            const uint32_t e = (ch * 4 + g) * 8 + l;
            o.xl[gg] = xt.xs[2 * e];
            o.xh[gg] = xt.xs[2 * e + 1];
            o.sum_lo[gg] = xt.sums[(ch * 4 + g) * 2];
            o.sum_hi[gg] = xt.sums[(ch * 4 + g) * 2 + 1];
        }
    }
    __device__ static void values(const PairChunk &k, const XC &xc, uint32_t hf, float (&c)[kNV]) {
        const float d = half_bits_to_float(k.s.x & 0xFFFFu);
        const float dmin = half_bits_to_float(k.s.x >> 16);
#pragma unroll
        for (uint32_t gg = 0; gg < 2; ++gg) {
            const float4 xl = xc.xl[gg], xh = xc.xh[gg];
            const float sum_lo = xc.sum_lo[gg], sum_hi = xc.sum_hi[gg];
            const uint32_t w = gg ? k.q.y : k.q.x;
            const uint32_t lo4 = w & 0x0F0F0F0Fu, hi4 = (w >> 4) & 0x0F0F0F0Fu;
            const float2 l01 = nibble_pair<false>(lo4), l23 = nibble_pair<true>(lo4);
            const float2 h01 = nibble_pair<false>(hi4), h23 = nibble_pair<true>(hi4);
            float alo = fma_rn(l01.x, xl.x, 0.0f);
            alo = fma_rn(l01.y, xl.y, alo);
            alo = fma_rn(l23.x, xl.z, alo);
            alo = fma_rn(l23.y, xl.w, alo);
            float ahi = fma_rn(h01.x, xh.x, 0.0f);
            ahi = fma_rn(h01.y, xh.y, ahi);
            ahi = fma_rn(h23.x, xh.z, ahi);
            ahi = fma_rn(h23.y, xh.w, ahi);
            const float hlo = hsum8_first(alo), hhi = hsum8_first(ahi);
            // sub-blocks 2 g and 2 g + 1 = 4 hf + 2 gg and 4 hf + 2 gg + 1
            uint32_t sc1, m1, sc2, m2;
            if (gg == 0) {
                scale_min<0>(k.s, hf, sc1, m1);
                scale_min<1>(k.s, hf, sc2, m2);
            } else {
                scale_min<2>(k.s, hf, sc1, m1);
                scale_min<3>(k.s, hf, sc2, m2);
            }
            const float dsc1 = d * static_cast<float>(sc1), dm1 = dmin * static_cast<float>(m1);
            const float dsc2 = d * static_cast<float>(sc2), dm2 = dmin * static_cast<float>(m2);
            const float part_lo = fma_rn(dsc1, hlo, -(dm1 * sum_lo));
            const float part_hi = fma_rn(dsc2, hhi, -(dm2 * sum_hi));
            c[gg] = part_lo + part_hi;
        }
    }
    // t = t + value for groups 0-3: own values, then the partner's.
    __device__ static float chain(const PairChunk &, const float (&c)[kNV], float t) {
        const float r0 = row_swap8(c[0]), r1 = row_swap8(c[1]);
        t = t + c[0];
        t = t + c[1];
        t = t + r0;
        return t + r1;
    }
    __device__ static float finish(float t) { return t; }
};

// The row's chunks in rings of PF + 1 register slots, chunk c + PF requested
// while chunk c is computed, and chunk c + 1's LDS operands read during chunk
// c's arithmetic (two operand sets, alternating with the slot's parity). The
// last one or two rings run with each request under a (wavefront-uniform)
// test, so nothing past the row's end is read.
template <class P, int PF>
__device__ __forceinline__ void pair_prime(const uint8_t *qp, const uint8_t *sp, uint32_t c_end,
                                           PairChunk (&buf)[PF + 1]) {
#pragma unroll
    for (int p = 0; p < PF; ++p) {
        const uint32_t c = static_cast<uint32_t>(p) < c_end ? p : c_end - 1;
        buf[p].q = ld8nt(qp + c * 128);
        buf[p].s = P::load_scales(sp + c * P::kScaleBytes);
    }
}

template <class P, int PF>
__device__ __forceinline__ float pair_stream(const uint8_t *qp, const uint8_t *sp, uint32_t c_end,
                                             const typename P::X &xt, uint32_t l, uint32_t hf,
                                             PairChunk (&buf)[PF + 1]) {
    constexpr uint32_t kSlots = PF + 1;
    static_assert(kSlots % 2 == 0, "the operand sets alternate with the parity of the ring slot");
    typename P::XC xc[2];
    P::read_x(xt, 0, l, hf, xc[0]);
    float t = 0.0f;
    uint32_t c = 0;
    for (; c + 2 * kSlots <= c_end; c += kSlots) {
#pragma unroll
        for (uint32_t p = 0; p < kSlots; ++p) {
            PairChunk &nx = buf[(p + PF) % kSlots];
            nx.q = ld8nt(qp + (p + PF) * 128);
            nx.s = P::load_scales(sp + (p + PF) * P::kScaleBytes);
            __builtin_amdgcn_sched_barrier(0);
            P::read_x(xt, c + p + 1, l, hf, xc[(p + 1) & 1]); // c + p + 1 < c_end in this loop
            float cv[P::kNV];
            P::values(buf[p], xc[p & 1], hf, cv);
            t = P::chain(buf[p], cv, t);
        }
        qp += kSlots * 128;
        sp += kSlots * P::kScaleBytes;
    }
    // the last chunks (fewer than two rings), in slot order
#pragma unroll
    for (uint32_t p = 0; p < 2 * kSlots; ++p) {
        if (c + p >= c_end) break;
        if (c + p + PF < c_end) {
            PairChunk &nx = buf[(p + PF) % kSlots];
            nx.q = ld8nt(qp + (p + PF) * 128);
            nx.s = P::load_scales(sp + (p + PF) * P::kScaleBytes);
        }
        if (c + p + 1 < c_end) P::read_x(xt, c + p + 1, l, hf, xc[(p + 1) & 1]);
        float cv[P::kNV];
        P::values(buf[p % kSlots], xc[p & 1], hf, cv);
        t = P::chain(buf[p % kSlots], cv, t);
    }
    return t;
}

} // namespace

} // namespace fmx
