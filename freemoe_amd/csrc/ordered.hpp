// ordered.hpp — sums of doubles in the reference's order, formed in parallel
// with a bound on their distance from the ordered sum.
#pragma once

#include "fmx_internal.hpp"

namespace fmx {

namespace {

// v moved across lanes by one DPP step; 0 where the step has no source lane.
template <int kCtrl, int kRows>
__device__ __forceinline__ double dpp_or_zero(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(b), kCtrl, kRows, 0xF, true);
    const uint32_t hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), kCtrl, kRows, 0xF, true);
    return __builtin_bit_cast(double, static_cast<uint64_t>(hi) << 32 | lo);
}

// Inclusive sum over the lanes of a wavefront: row_shr:1, 2, 4, 8 inside the
// rows of 16, then lane 15 of each even row into the odd row after it, then
// lane 31 into the upper half.
__device__ __forceinline__ double wave_scan(double v) {
    v += dpp_or_zero<0x111, 0xF>(v);
    v += dpp_or_zero<0x112, 0xF>(v);
    v += dpp_or_zero<0x114, 0xF>(v);
    v += dpp_or_zero<0x118, 0xF>(v);
    v += dpp_or_zero<0x142, 0xA>(v);
    v += dpp_or_zero<0x143, 0xC>(v);
    return v;
}

__device__ __forceinline__ double last_lane(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = __builtin_amdgcn_readlane(static_cast<int>(b), 63);
    const uint32_t hi = __builtin_amdgcn_readlane(static_cast<int>(b >> 32), 63);
    return __builtin_bit_cast(double, static_cast<uint64_t>(hi) << 32 | lo);
}

__device__ __forceinline__ double wave_sum(double v) { return last_lane(wave_scan(v)); }

__device__ __forceinline__ uint32_t exponent_of(double v) {
    return static_cast<uint32_t>(__builtin_bit_cast(uint64_t, v) >> 52);
}
__device__ __forceinline__ double power_of(uint32_t exponent) { // 0 below the normal range
    return __builtin_bit_cast(double, static_cast<uint64_t>(exponent) << 52);
}

// hi + lo += v, exactly but for the last rounding of lo.
__device__ __forceinline__ void add_exact(double &hi, double &lo, double v, double v_lo = 0.0) {
    const double s = hi + v, b = s - hi;
    lo += ((hi - (s - b)) + (v - b)) + v_lo;
    hi = s;
}

// The sum of a workgroup's terms in order, s_t = rn(s_t-1 + x_t) from 0, to
// within `doubt`: thread i adds the terms after thread i - 1's, from the
// (unordered) sum `run` of those before, which no ordered prefix sum is
// further from than `margin`. While s stays in one binade, of unit u, a step
// adds x_t rounded to a multiple of u, whatever s is, but for exact ties; so
// where the margin leaves no doubt about the binades of s_t-1 and s_t, the
// step is known but for half a unit at a tie, and elsewhere to within a unit.
// x_t has at most 48 significant bits or is no larger in magnitude than s_t.
struct OrderedInterval {
    double run, margin;
    double hi = 0.0, lo = 0.0, unc = 0.0;

    __device__ __forceinline__ void add(double x) {
        const double after = run + x;
        const uint32_t k = exponent_of(fabs(after) + margin);
        const double u = power_of(k > 52 ? k - 52 : 0);
        double r = x;
        if (exponent_of(fabs(after) - margin) != k || fabs(run) <= margin || exponent_of(fabs(run) - margin) < k) {
            unc += u;
        } else if (fabs(x) < power_of(k)) { // else a multiple of u
            const double big = copysign(power_of(k), x);
            r = (big + x) - big;
            if (fabs(x - r) * 2.0 == u) {
                r = x;
                unc += 0.5 * u;
            }
        }
        add_exact(hi, lo, r);
        run = after;
    }

    // After the thread's last term. Every thread returns the same sum; red: 3 x
    // kWaves doubles of LDS.
    template <uint32_t kWaves>
    __device__ __forceinline__ void total(double (&red)[3][kWaves], double &sum, double &doubt) {
        auto wave_total = [&] {
            add_exact(hi, lo, dpp_or_zero<0x111, 0xF>(hi), dpp_or_zero<0x111, 0xF>(lo));
            add_exact(hi, lo, dpp_or_zero<0x112, 0xF>(hi), dpp_or_zero<0x112, 0xF>(lo));
            add_exact(hi, lo, dpp_or_zero<0x114, 0xF>(hi), dpp_or_zero<0x114, 0xF>(lo));
            add_exact(hi, lo, dpp_or_zero<0x118, 0xF>(hi), dpp_or_zero<0x118, 0xF>(lo));
            add_exact(hi, lo, dpp_or_zero<0x142, 0xA>(hi), dpp_or_zero<0x142, 0xA>(lo));
            add_exact(hi, lo, dpp_or_zero<0x143, 0xC>(hi), dpp_or_zero<0x143, 0xC>(lo));
            hi = last_lane(hi);
            lo = last_lane(lo);
            unc = wave_sum(unc);
        };
        wave_total();
        const uint32_t lane = threadIdx.x & 63;
        if (lane == 0) {
            red[0][threadIdx.x >> 6] = hi;
            red[1][threadIdx.x >> 6] = lo;
            red[2][threadIdx.x >> 6] = unc;
        }
        __syncthreads();
        hi = lane < kWaves ? red[0][lane] : 0.0;
        lo = lane < kWaves ? red[1][lane] : 0.0;
        unc = lane < kWaves ? red[2][lane] : 0.0;
        wave_total();
        sum = hi + lo;
        // the bound's own roundings, and the sum's
        doubt = unc * 1.0009765625 + fabs(sum) * 0x1p-52 + margin * 0x1p-40;
    }
};

// OrderedInterval over the first nt <= kTerms of a thread's terms.
template <uint32_t kTerms, uint32_t kWaves>
__device__ __forceinline__ void ordered_interval(const double (&x)[kTerms], uint32_t nt, double run, double margin,
                                                 double (&red)[3][kWaves], double &sum, double &doubt) {
    OrderedInterval s{run, margin};
#pragma unroll
    for (uint32_t i = 0; i < kTerms; ++i)
        if (i < nt) s.add(x[i]);
    s.total(red, sum, doubt);
}

} // namespace

} // namespace fmx
