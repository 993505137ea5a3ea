// attention.hip — one token's decode attention over its cached positions
// (FreeMoe's engine.cpp:1360-1420, the full-context MHA / GQA case) on
// gfx950, for fm::HipBackend::attention.
//
// Per query head h (kv head h / (heads / kv_heads)), over cached positions
// t = 0 .. P-1:
//   s_t   = float(dot(q_h, k_t) * scale), the dot a double sum over the head
//           dimension in index order (a float times a float is exact in
//           double, so every rounding is the engine's);
//   p     = the engine's softmax of s (engine.cpp:378-393): the float
//           maximum m, e_t = exp(double(s_t) - m), their double sum in
//           position order, p_t = float(e_t / sum);
//   out_j = float(sum_t double(p_t) v_t[j]) in position order.
// Only exp is the device's own (the engine calls the host libm's); both are
// within an ulp, so a result can differ in its last bit where a value sits
// on a rounding boundary. A non-finite score (the engine raises
// INTERNAL_ERROR) sets bit 0 of the status word.
//
// Both sums over the positions are formed in parallel with a bound on how far
// the sum in position order can lie from the parallel one. A probability or
// an output whose float is the same over that whole interval is the engine's;
// where one is not, one lane adds the terms in order. For 32 heads of 128 over
// 8 kv heads and 2000 positions (16 MB of cache: 3 us of HBM) a call takes 20
// us, three dependent launches (traced one by one: 1, 6 and 14 us), each a
// chain of memory, LDS and double-precision latencies; walking every sum in
// order on one workgroup per head took 215 us (32 of the 256 CUs in use). 8192
// positions: 46 us, 83 over 32 kv heads.
#include <atomic>

#include "fmx_internal.hpp"
#include "ordered.hpp"

namespace fmx {

namespace {

constexpr uint32_t kCus = 256;
constexpr uint32_t kMaxHeadDim = 256;
constexpr uint32_t kMaxPositions = 8192;
constexpr uint32_t kScorePos = 32;  // positions of a score workgroup
constexpr uint32_t kScoreHeads = 4; // heads it scores at a time
constexpr uint32_t kSliceDims = 16; // output elements of a value workgroup
constexpr uint32_t kGroupPad = 4;   // its LDS rows of group sums: the four columns' stores on other banks

// Up to this many positions every slice's workgroup computes the scores of its
// head itself, one per thread: 32 heads of 128 over 256 positions 11.4 us, over
// 257, with the score kernel's launch before it, 14.4 (at 512, two per thread,
// no faster).
constexpr uint32_t kSplitPositions = 256;

// Scores between the two kernels of a call: kSlots buffers of device memory,
// taken in turn. Nothing holds a buffer: a score carries its call's ticket, and
// a value workgroup that finds another's among its head's (more than kSlots
// calls in flight, or a replayed graph's fixed ticket meeting another call's)
// computes them all itself. So a call never reads another's scores, whatever
// runs beside it; executions of one captured call share a ticket, and with it
// the inputs the scores come from. (Four buffers: as many calls as a process
// has hardware queues run at once.)
constexpr uint32_t kSlots = 4;
constexpr uint32_t kSlotScores = 512 * 1024;
__device__ __align__(256) uint64_t slot_scores[kSlots][kSlotScores];

// One access each, so that a score and its ticket stay together.
__device__ __forceinline__ void put_score(uint64_t *at, float score, uint32_t ticket) {
    __hip_atomic_store(at, static_cast<uint64_t>(ticket) << 32 | __builtin_bit_cast(uint32_t, score), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t get_score(const uint64_t *at) {
    return __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ void attention_clear_kernel(uint32_t *status) { *status = 0; }

// The dot of one key with one query (doubles in LDS), in index order. fma:
// the product is exact, so it rounds once, as the engine's multiply and add.
__device__ __forceinline__ double dot_in_order(const float *k, const double *q, uint32_t head_dim) {
    double dot = 0.0;
#pragma unroll 8
    for (uint32_t j = 0; j < head_dim; j += 4) {
        const float4 v = *reinterpret_cast<const float4 *>(k + j);
        const double2 a = *reinterpret_cast<const double2 *>(q + j);
        const double2 b = *reinterpret_cast<const double2 *>(q + j + 2);
        dot = fma(a.x, static_cast<double>(v.x), dot);
        dot = fma(a.y, static_cast<double>(v.y), dot);
        dot = fma(b.x, static_cast<double>(v.z), dot);
        dot = fma(b.y, static_cast<double>(v.w), dot);
    }
    return dot;
}

// Scores of 32 positions for every query head of one kv head, into the
// ticket's slot. The keys are read once, whole rows at a time, into LDS (rows 4
// floats apart in banks); a lane runs one (position, head) chain of head_dim
// fmas.
// grid: position tiles x kv heads; LDS: keys, then 4 heads' queries.
__global__ __launch_bounds__(kScorePos *kScoreHeads) void attention_scores_kernel(
    const float *__restrict__ q, const float *__restrict__ kv, uint64_t row_stride, uint32_t group,
    uint32_t head_dim, uint32_t positions, double scale, uint32_t ticket) {
    extern __shared__ __align__(16) char lds[];
    const uint32_t tid = threadIdx.x, kvh = blockIdx.y, t0 = blockIdx.x * kScorePos;
    const uint32_t kstride = head_dim + 4, qstride = head_dim + 2, D4 = head_dim / 4;
    float *ks = reinterpret_cast<float *>(lds);
    double *qs = reinterpret_cast<double *>(ks + kScorePos * kstride);
    const float *keys = kv + static_cast<uint64_t>(kvh) * head_dim;
#pragma unroll 8
    for (uint32_t i = tid; i < kScorePos * D4; i += kScorePos * kScoreHeads) {
        const uint32_t p = i / D4, j = i % D4;
        const uint32_t t = t0 + p < positions ? t0 + p : positions - 1; // clamp: loads stay in the cache
        *reinterpret_cast<float4 *>(ks + p * kstride + 4 * j) =
            *reinterpret_cast<const float4 *>(keys + t * row_stride + 4 * j);
    }
    const uint32_t pos = tid % kScorePos, hs = tid / kScorePos;
    uint64_t *dst = slot_scores[ticket % kSlots] + t0 + pos;
    for (uint32_t h0 = 0; h0 < group; h0 += kScoreHeads) {
        const uint32_t nh = group - h0 < kScoreHeads ? group - h0 : kScoreHeads;
        const uint64_t head0 = static_cast<uint64_t>(kvh) * group + h0;
        if (h0) __syncthreads();
        for (uint32_t i = tid; i < nh * head_dim; i += kScorePos * kScoreHeads)
            qs[i / head_dim * qstride + i % head_dim] = static_cast<double>(q[head0 * head_dim + i]);
        __syncthreads();
        if (hs < nh && t0 + pos < positions)
            put_score(dst + (head0 + hs) * positions,
                      static_cast<float>(dot_in_order(ks + pos * kstride, qs + hs * qstride, head_dim) * scale), ticket);
    }
}

// s + a[0] + a[1] + ... in order, for one lane: the next 16 terms are read
// from LDS during the current 16's additions.
__device__ __forceinline__ double add_in_order(const double *a, uint32_t n, double s) {
    constexpr uint32_t kBatch = 16;
    double cur[kBatch], next[kBatch];
    const uint32_t full = n / kBatch * kBatch;
    if (full) {
#pragma unroll
        for (uint32_t i = 0; i < kBatch; ++i) cur[i] = a[i];
    }
    for (uint32_t t = 0; t < full; t += kBatch) {
        const double *from = a + (t + kBatch < full ? t + kBatch : t);
#pragma unroll
        for (uint32_t i = 0; i < kBatch; ++i) next[i] = from[i];
#pragma unroll
        for (uint32_t i = 0; i < kBatch; ++i) s += cur[i];
#pragma unroll
        for (uint32_t i = 0; i < kBatch; ++i) cur[i] = next[i];
    }
    for (uint32_t t = full; t < n; ++t) s += a[t];
    return s;
}

// grid: heads x slices of 16 output elements. LDS: positions doubles (the
// exponentials where they are added in order; otherwise the probabilities as
// floats), then the value sums of NT / 4 position groups.
//
// Softmax: every slice's workgroup repeats its head's, on NT threads of up to
// kTerms consecutive positions. The sum of the exponentials in order is known
// to a few units in 2^53 (ordered_interval), so all but about one of 2^23
// probabilities are decided.
//
// Values: thread (g, c) sums its group's consecutive positions for four
// elements; the sum in position order differs from theirs by at most the
// roundings of its partial sums, each bounded by the prefix of the group it
// is in plus the group's absolute sum. That decides all but about one of 10^5
// elements (at 2000 positions; one of 10^4 at 8192); ordered_interval over
// the element's products nearly all of the rest.
template <uint32_t NT, uint32_t kTerms>
__global__ __launch_bounds__(NT) void attention_values_kernel(
    const float *__restrict__ q, const float *__restrict__ kv, uint64_t row_stride, uint32_t v_offset,
    uint32_t heads, uint32_t group, uint32_t head_dim, uint32_t positions, double scale, float *__restrict__ out,
    uint32_t *__restrict__ status, uint32_t ticket) {
    constexpr uint32_t kWaves = NT / 64, kGroups = NT / (kSliceDims / 4);
    constexpr uint32_t kPrefetch = kTerms > 2 ? 4 : 8; // (8 beside eight terms spill)
    constexpr uint32_t kGroupStride = kGroups + kGroupPad;
    extern __shared__ __align__(16) char lds[];
    __shared__ __align__(16) double qs[kMaxHeadDim];
    __shared__ float red_max[kWaves];
    __shared__ double red_sum[kWaves], red[3][kWaves], err_s[kSliceDims];
    __shared__ bool stale_s[kWaves];
    __shared__ uint32_t flags_s, todo_s; // 1: non-finite score, 2: a probability undecided
    __shared__ double sum_s;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t P = positions, D = head_dim;
    const uint32_t slices = div_up(D, kSliceDims), total = heads * slices;
    // workgroup i runs on XCD i % 8: give each XCD consecutive heads, so that
    // the heads of a kv head read its values through one L2
    const uint32_t unit = total % 8 == 0 ? blockIdx.x % 8 * (total / 8) + blockIdx.x / 8 : blockIdx.x;
    const uint32_t head = unit / slices, slice = unit % slices, kvh = head / group;
    double *ex = reinterpret_cast<double *>(lds);
    float *pr = reinterpret_cast<float *>(lds);
    double *gsum = reinterpret_cast<double *>(lds + ((static_cast<size_t>(P) * 8 + 15) & ~static_cast<size_t>(15)));
    float *gabs = reinterpret_cast<float *>(gsum + kSliceDims * kGroupStride);

    // the head's scores, then the first positions of this thread's values, which
    // stay in flight during the softmax
    uint64_t raw[kTerms];
    if (ticket != 0) {
        const uint64_t *src = slot_scores[ticket % kSlots] + static_cast<uint64_t>(head) * P;
#pragma unroll
        for (uint32_t i = 0; i < kTerms; ++i) raw[i] = get_score(src + (i * NT + tid < P ? i * NT + tid : P - 1));
    }
    const uint32_t col = slice * kSliceDims + (tid & 3) * 4, grp = tid >> 2;
    const uint32_t per_group = div_up(P, kGroups);
    const uint32_t v0 = grp * per_group < P ? grp * per_group : P;
    const uint32_t v1 = v0 + per_group < P ? v0 + per_group : P;
    const float *vbase = kv + v_offset + static_cast<uint64_t>(kvh) * D + (col < D ? col : 0);
    float4 vv[kPrefetch];
#pragma unroll
    for (uint32_t i = 0; i < kPrefetch; ++i) {
        const uint32_t t = v0 + i < P ? v0 + i : P - 1;
        vv[i] = *reinterpret_cast<const float4 *>(vbase + t * row_stride);
    }

    // scores t0 .. t1 - 1 of this thread
    const uint32_t per = div_up(P, NT);
    const uint32_t t0 = tid * per < P ? tid * per : P;
    const uint32_t nt = t0 + per < P ? per : P - t0;
    bool stale = ticket == 0;
    if (!stale) {
#pragma unroll
        for (uint32_t i = 0; i < kTerms; ++i)
            if (i * NT + tid < P) {
                pr[i * NT + tid] = __builtin_bit_cast(float, static_cast<uint32_t>(raw[i]));
                stale |= static_cast<uint32_t>(raw[i] >> 32) != ticket;
            }
    }
    stale = __any(stale);
    if (lane == 0) stale_s[wave] = stale;
    if (tid == 0) flags_s = todo_s = 0;
    __syncthreads();
#pragma unroll
    for (uint32_t i = 0; i < kWaves; ++i) stale |= stale_s[i];
    float sc[kTerms];
    if (!stale) {
#pragma unroll
        for (uint32_t i = 0; i < kTerms; ++i)
            if (i < nt) sc[i] = pr[t0 + i];
    } else {
        for (uint32_t j = tid; j < D; j += NT) qs[j] = static_cast<double>(q[static_cast<uint64_t>(head) * D + j]);
        __syncthreads();
#pragma unroll
        for (uint32_t i = 0; i < kTerms; ++i)
            if (i < nt)
                sc[i] = static_cast<float>(
                    dot_in_order(kv + (t0 + i) * row_stride + static_cast<uint64_t>(kvh) * D, qs, D) * scale);
    }
    float m = -__builtin_inff();
    bool bad = false;
#pragma unroll
    for (uint32_t i = 0; i < kTerms; ++i)
        if (i < nt) {
            bad |= !__builtin_isfinite(sc[i]);
            m = fmaxf(m, sc[i]);
        }
    for (uint32_t d = 32; d >= 1; d >>= 1) m = fmaxf(m, __shfl_xor(m, d));
    if (lane == 0) red_max[wave] = m;
    __syncthreads();
    if (__any(bad) && lane == 0) atomicOr(&flags_s, 1u);
#pragma unroll
    for (uint32_t i = 0; i < kWaves; ++i) m = fmaxf(m, red_max[i]);
    const double md = static_cast<double>(m);
    double e[kTerms], local = 0.0;
#pragma unroll
    for (uint32_t i = 0; i < kTerms; ++i) {
        e[i] = i < nt ? exp(static_cast<double>(sc[i]) - md) : 0.0;
        local += e[i];
    }
    const double incl = wave_scan(local);
    if (lane == 63) red_sum[wave] = incl;
    __syncthreads();
    if (flags_s & 1u) {
        if (tid == 0 && slice == 0) atomicOr(status, STATUS_NONFINITE_SCORE);
        if (tid < 4 && col < D)
            *reinterpret_cast<float4 *>(out + static_cast<uint64_t>(head) * D + col) = make_float4(0.f, 0.f, 0.f, 0.f);
        return;
    }
    double run = incl - local, all = 0.0;
#pragma unroll
    for (uint32_t i = 0; i < kWaves; ++i) {
        run += i < wave ? red_sum[i] : 0.0;
        all += red_sum[i];
    }
    // (an ordered prefix sum is off by at most P 2^-53 of the whole, run by
    // 30 2^-53)
    double sum, doubt;
    ordered_interval(e, nt, run, all * 0x1p-38, red, sum, doubt);
    // relative: the doubt, the roundings of the reciprocal, of the products
    // below and of the engine's division
    const double rinv = 1.0 / sum, rel = doubt * rinv * 1.0009765625 + 0x1p-50;
    float p[kTerms];
    bool undecided = !(rel < 0x1p-30);
#pragma unroll
    for (uint32_t i = 0; i < kTerms; ++i)
        if (i < nt) {
            const double v = e[i] * rinv;
            p[i] = static_cast<float>(v - v * rel);
            undecided |= p[i] != static_cast<float>(v + v * rel);
        }
    if (__any(undecided) && lane == 0) atomicOr(&flags_s, 2u);
    __syncthreads();
    if (flags_s & 2u) { // the exponentials added in order by one lane
#pragma unroll
        for (uint32_t i = 0; i < kTerms; ++i)
            if (i < nt) ex[t0 + i] = e[i];
        __syncthreads();
        if (tid == 0) sum_s = add_in_order(ex, P, 0.0);
        __syncthreads();
        const double s = sum_s;
#pragma unroll
        for (uint32_t i = 0; i < kTerms; ++i)
            if (i < nt) p[i] = static_cast<float>(e[i] / s);
    }
#pragma unroll
    for (uint32_t i = 0; i < kTerms; ++i)
        if (i < nt) pr[t0 + i] = p[i];
    __syncthreads();

    // values: this thread's positions of its group, four elements
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    float aabs[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t tb = v0; tb < v1; tb += kPrefetch) {
        float4 cur[kPrefetch];
#pragma unroll
        for (uint32_t i = 0; i < kPrefetch; ++i) {
            cur[i] = vv[i];
            const uint32_t t = tb + kPrefetch + i < P ? tb + kPrefetch + i : P - 1;
            if (tb + kPrefetch < v1) vv[i] = *reinterpret_cast<const float4 *>(vbase + t * row_stride);
        }
#pragma unroll
        for (uint32_t i = 0; i < kPrefetch; ++i)
            if (tb + i < v1) {
                const float w = pr[tb + i];
                const double wd = static_cast<double>(w);
                const float x[4] = {cur[i].x, cur[i].y, cur[i].z, cur[i].w};
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) {
                    acc[j] = fma(wd, static_cast<double>(x[j]), acc[j]);
                    aabs[j] = fma_rn(w, fabsf(x[j]), aabs[j]);
                }
            }
    }
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
        gsum[((tid & 3) * 4 + j) * kGroupStride + grp] = acc[j];
        gabs[((tid & 3) * 4 + j) * kGroupStride + grp] = aabs[j];
    }
    __syncthreads();
    // a wavefront takes kPerWave elements: prefix sums of the groups and the bound
    constexpr uint32_t kPerLane = kGroups / 64, kPerWave = kSliceDims / kWaves;
#pragma unroll
    for (uint32_t i = 0; i < kPerWave; ++i) {
        const uint32_t d = wave * kPerWave + i;
        double gs[kPerLane], ga[kPerLane], s = 0.0, a = 0.0;
#pragma unroll
        for (uint32_t k = 0; k < kPerLane; ++k) {
            gs[k] = gsum[d * kGroupStride + lane * kPerLane + k];
            // (the float sum's own error, and products below float's range)
            ga[k] = static_cast<double>(gabs[d * kGroupStride + lane * kPerLane + k]) * 1.0009765625 + 0x1p-120;
            s += gs[k];
            a += ga[k];
        }
        const double scan = wave_scan(s);
        double before = scan - s, bound = 0.0;
#pragma unroll
        for (uint32_t k = 0; k < kPerLane; ++k) {
            bound += fabs(before) + ga[k];
            before += gs[k];
        }
        // per_group roundings of partial sums no larger than |before| + ga,
        // as many here of sums no larger than ga, and the tree's (of at most
        // a each): each 2^-53 of its sum, and a sixteenth for the bounds' own
        // roundings
        const double value = last_lane(scan);
        const double err = wave_sum(per_group * (bound + a) + 16.0 * a) * 0x1.1p-53;
        const float lo = static_cast<float>(value - err), hi = static_cast<float>(value + err);
        const uint32_t j = slice * kSliceDims + d;
        if (lane == 0 && j < D) {
            if (__builtin_bit_cast(uint32_t, lo) == __builtin_bit_cast(uint32_t, hi) && __builtin_isfinite(lo))
                out[static_cast<uint64_t>(head) * D + j] = lo;
            else {
                atomicOr(&todo_s, 1u << d);
                err_s[d] = err;
            }
        }
    }
    __syncthreads();
    // the elements left: by the intervals of their products (exact in
    // double), then in position order, the products in LDS and one lane adding
    constexpr uint32_t kTile = kSliceDims * kGroupStride;
    for (uint32_t todo = todo_s; todo; todo &= todo - 1) {
        const uint32_t d = __builtin_ctz(todo), j = slice * kSliceDims + d;
        const float *v = kv + v_offset + static_cast<uint64_t>(kvh) * D + j;
        double x[kTerms], before = 0.0;
#pragma unroll
        for (uint32_t i = 0; i < kTerms; ++i) {
            x[i] = i < nt ? static_cast<double>(p[i]) * static_cast<double>(v[(t0 + i) * row_stride]) : 0.0;
            before += x[i];
        }
        const double mine = before, scan = wave_scan(mine);
        if (lane == 63) red_sum[wave] = scan;
        __syncthreads();
        before = scan - mine;
#pragma unroll
        for (uint32_t i = 0; i < kWaves; ++i) before += i < wave ? red_sum[i] : 0.0;
        // (err_s bounds the ordered sum's roundings and 17 2^-53 of the
        // absolute sum; these prefixes' add up to 30 of them)
        double s, off;
        ordered_interval(x, nt, before, 3.0 * err_s[d], red, s, off);
        const float lo = static_cast<float>(s - off), hi = static_cast<float>(s + off);
        if (__builtin_bit_cast(uint32_t, lo) == __builtin_bit_cast(uint32_t, hi) && __builtin_isfinite(lo)) {
            if (tid == 0) out[static_cast<uint64_t>(head) * D + j] = lo;
            __syncthreads(); // red_sum and red are read
            continue;
        }
        s = 0.0;
        for (uint32_t tb = 0; tb < P; tb += kTile) {
            const uint32_t n = P - tb < kTile ? P - tb : kTile;
            for (uint32_t i = tid; i < n; i += NT)
                gsum[i] = static_cast<double>(pr[tb + i]) * static_cast<double>(v[(tb + i) * row_stride]);
            __syncthreads();
            if (tid == 0) s = add_in_order(gsum, n, s);
            __syncthreads();
        }
        if (tid == 0) out[static_cast<uint64_t>(head) * D + j] = static_cast<float>(s);
    }
}

// A head's whole attention on one workgroup, every sum in order: a launch with
// nothing repeated between workgroups (attention_values_kernel repeats the
// softmax in every slice, and its 1024 threads have a CU to themselves).
// grid: heads; LDS: positions doubles, then as many floats.
constexpr uint32_t kHeadThreads = 256;
__global__ __launch_bounds__(kHeadThreads) void attention_heads_kernel(
    const float *__restrict__ q, const float *__restrict__ kv, uint64_t row_stride, uint32_t v_offset, uint32_t group,
    uint32_t head_dim, uint32_t positions, double scale, float *__restrict__ out, uint32_t *__restrict__ status) {
    constexpr uint32_t kWaves = kHeadThreads / 64;
    extern __shared__ __align__(16) char lds[];
    __shared__ __align__(16) double qs[kMaxHeadDim];
    __shared__ float red_max[kWaves];
    __shared__ bool bad_s[kWaves];
    __shared__ double sum_s;
    const uint32_t tid = threadIdx.x, wave = tid >> 6, head = blockIdx.x, P = positions, D = head_dim;
    double *ex = reinterpret_cast<double *>(lds);
    float *pr = reinterpret_cast<float *>(ex + P);
    const float *keys = kv + static_cast<uint64_t>(head / group) * D;
    float *o = out + static_cast<uint64_t>(head) * D;
    if (tid < D) qs[tid] = static_cast<double>(q[static_cast<uint64_t>(head) * D + tid]);
    __syncthreads();
    float m = -__builtin_inff();
    bool bad = false;
    for (uint32_t t = tid; t < P; t += kHeadThreads) {
        const float s = static_cast<float>(dot_in_order(keys + t * row_stride, qs, D) * scale);
        bad |= !__builtin_isfinite(s);
        m = fmaxf(m, s);
        pr[t] = s;
    }
    for (uint32_t d = 32; d >= 1; d >>= 1) m = fmaxf(m, __shfl_xor(m, d));
    bad = __any(bad);
    if ((tid & 63) == 0) {
        red_max[wave] = m;
        bad_s[wave] = bad;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t i = 0; i < kWaves; ++i) {
        m = fmaxf(m, red_max[i]);
        bad |= bad_s[i];
    }
    if (bad) {
        if (tid == 0) atomicOr(status, STATUS_NONFINITE_SCORE);
        if (tid < D) o[tid] = 0.0f;
        return;
    }
    const double md = static_cast<double>(m);
    for (uint32_t t = tid; t < P; t += kHeadThreads) ex[t] = exp(static_cast<double>(pr[t]) - md);
    __syncthreads();
    if (tid == 0) sum_s = add_in_order(ex, P, 0.0);
    __syncthreads();
    const double sum = sum_s;
    for (uint32_t t = tid; t < P; t += kHeadThreads) pr[t] = static_cast<float>(ex[t] / sum);
    __syncthreads();
    if (tid >= D) return;
    const float *v = keys + v_offset + tid;
    double acc = 0.0; // fma: the product is exact
#pragma unroll 8
    for (uint32_t t = 0; t < P; ++t)
        acc = fma(static_cast<double>(pr[t]), static_cast<double>(v[t * row_stride]), acc);
    o[tid] = static_cast<float>(acc);
}

size_t values_lds_bytes(uint32_t positions, uint32_t threads) {
    return ((static_cast<size_t>(positions) * 8 + 15) & ~static_cast<size_t>(15)) + (threads / 4 + kGroupPad) * kSliceDims * 12;
}

// Whether a call of `total` slices takes attention_heads_kernel. A slice's
// workgroup of 1024 threads fills a CU: up to 256 slices run at once, and only
// the shortest caches are better off on one workgroup per head; beyond, the
// slices come in rounds while the heads do not. Heads x kv heads x dim x
// positions, heads kernel / slices, us: 32 x 4 x 128 x 16 7.1 / 8.9, x 64 8.5 /
// 9.0, x 96 9.6 / 9.2; 64 x 64 x 128 x 256 15.0 / 16.2, x 400 21.7 / 23.6, x 512
// 28.9 / 25.1; 128 x 128 x 256 x 256 26 / 68, x 1024 96 / 127, x 1536 192 / 176.
// Where the scores do not fit a buffer every slice forms its head's: 256 x 32 x
// 128 x 3000 191 / 469, but 128 x 128 x 128 x 8192 (1024 slices) about 1100 /
// 760. Over 1800 such calls the rule's choice never costs more than 21% over
// the other's time.
bool attention_on_heads(uint32_t heads, uint32_t total, uint32_t positions) {
    if (total <= kCus) return positions < 72;
    if (positions > kSplitPositions && static_cast<uint64_t>(heads) * positions > kSlotScores) return total > 1024;
    return positions < 450 || positions < total * 11 / 20;
}

// A call's ticket: never 0, and its slot modulo kSlots.
uint32_t next_ticket() {
    static std::atomic<uint32_t> counter{0};
    uint32_t t;
    do t = counter.fetch_add(1, std::memory_order_relaxed) + 1;
    while (t == 0);
    return t;
}

} // namespace

int attention_decode(const float *q, const float *kv, uint64_t row_stride, uint32_t v_offset, uint32_t heads,
                     uint32_t kv_heads, uint32_t head_dim, uint32_t positions, double scale, float *out,
                     uint32_t *status, hipStream_t s) {
    if (heads == 0 || kv_heads == 0 || heads % kv_heads || head_dim == 0 || head_dim > kMaxHeadDim ||
        head_dim % 4 || positions == 0 || positions > kMaxPositions || row_stride % 4 || v_offset % 4)
        return FMX_ERR_SHAPE_MISMATCH;
    if (v_offset + static_cast<uint64_t>(kv_heads) * head_dim > row_stride ||
        static_cast<uint64_t>(kv_heads) * head_dim > v_offset)
        return FMX_ERR_SHAPE_MISMATCH;
    const uint32_t group = heads / kv_heads;
    const uint32_t total = heads * div_up(head_dim, kSliceDims);
    if (attention_on_heads(heads, total, positions)) {
        const size_t lds = static_cast<size_t>(positions) * 12;
        if (int rc = allow_lds(reinterpret_cast<const void *>(attention_heads_kernel), lds)) return rc;
        hipLaunchKernelGGL(attention_clear_kernel, dim3(1), dim3(1), 0, s, status);
        FMX_LAUNCH_CHECK();
        hipLaunchKernelGGL(attention_heads_kernel, dim3(heads), dim3(kHeadThreads), lds, s, q, kv, row_stride, v_offset,
                           group, head_dim, positions, scale, out, status);
        FMX_LAUNCH_CHECK();
        return FMX_OK;
    }
    const bool split = positions > kSplitPositions && static_cast<uint64_t>(heads) * positions <= kSlotScores &&
                       kv_heads <= 65535;
    const uint32_t ticket = split ? next_ticket() : 0;
    // as few terms per thread as the threads allow: their exponentials and
    // divisions are one after another
    const auto values = positions <= 256    ? attention_values_kernel<256, 1>
                        : positions <= 2048 ? attention_values_kernel<1024, 2>
                                            : attention_values_kernel<1024, 8>;
    const uint32_t threads = positions <= 256 ? 256 : 1024;
    const size_t lds = values_lds_bytes(positions, threads);
    if (int rc = allow_lds(reinterpret_cast<const void *>(values), lds)) return rc;
    hipLaunchKernelGGL(attention_clear_kernel, dim3(1), dim3(1), 0, s, status);
    FMX_LAUNCH_CHECK();
    if (split) {
        const size_t tile = kScorePos * (head_dim + 4) * sizeof(float) + kScoreHeads * (head_dim + 2) * sizeof(double);
        hipLaunchKernelGGL(attention_scores_kernel, dim3(div_up(positions, kScorePos), kv_heads),
                           dim3(kScorePos * kScoreHeads), tile, s, q, kv, row_stride, group, head_dim, positions,
                           scale, ticket);
        FMX_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(values, dim3(total), dim3(threads), lds, s, q, kv, row_stride, v_offset, heads, group, head_dim,
                       positions, scale, out, status, ticket);
    FMX_LAUNCH_CHECK();
    return FMX_OK;
}

} // namespace fmx
