// k_sampling.hip — greedy arg-max and top-k / temperature / top-p sampling.
//
// Replaces topk_temperature_softmax_sampling_kernel_bf16 + blockArgMax/better
// (layers/src/logit_decode.cu:15-33, 149-274) and sample_topk_bf16
// (helpers.cuh:157-166).  The reference runs ONE 256-thread block that makes k
// full sweeps over V with an O(k) membership scan per element.  Here:
//   * every logit maps to a 64-bit selection key whose order IS the reference's
//     selection order (value, then bitrev8(idx mod 256), then -idx; see
//     qie_common.hpp sel_key) — greedy is a parallel max over keys (also fused
//     into the lm_head GEMV epilogue, k_gemv.hip);
//   * top-k = a radix selection per 4096-slice, sorted, and one pass over the slices' winners that
//     leaves out what cannot be among the k; the sorted keys reproduce the reference's k rounds exactly;
//   * softmax + draw in one wave: exponentials a lane each, sums in the reference's
//     sequential order lane by lane, and a cuRAND-XORWOW restatement (curand_init(seed, 0, 0);
//     curand_uniform).
#include "qie_common.hpp"
#include "../../include/qie/qie_ops.h"

namespace qie {

constexpr int kSlice = 4096;
constexpr int kMaxTopK = 256;

__global__ __launch_bounds__(256) void argmax_keys_kernel(const uint16_t* __restrict__ logits,
                                                          int64_t V, int64_t ld,
                                                          unsigned long long* keys) {
    __shared__ unsigned long long red[4];
    const int64_t m = blockIdx.y;
    const uint16_t* row = logits + m * ld;
    unsigned long long best = 0ull;
    const int64_t per = (V + gridDim.x - 1) / gridDim.x;
    const int64_t lo = blockIdx.x * per, hi = min(V, lo + per);
    for (int64_t i = lo + threadIdx.x; i < hi; i += 256) {
        unsigned long long k = sel_key(bf2f(row[i]), (uint32_t)i);
        best = k > best ? k : best;
    }
    best = wave_max(best);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long b = red[0];
        for (int w = 1; w < 4; w++) b = red[w] > b ? red[w] : b;
        if (b) atomicMax(keys + m, b);
    }
}

__global__ void keys_to_ids_kernel(const unsigned long long* keys, int64_t M, int32_t* ids) {
    const int64_t m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m < M) ids[m] = key_idx(keys[m]);
}

// The k largest of a block's keys (KPT a thread, in registers), unordered, into out[0, k) (LDS or memory; zeros behind the
// last where fewer than k keys are non-zero).  Radix selection from the top byte: a histogram of the keys that still share the
// threshold's prefix, until the bin of the k-th holds just what is needed: three to six passes of about 1.5 us.  (Bits 47..32 are the low half of a bf16's fp32 pattern: known from its sign.)
template <int KPT>
__device__ void radix_top(const unsigned long long (&key)[KPT], int k, unsigned long long* out) {
    __shared__ unsigned hist[256];
    __shared__ unsigned pick[3];   // digit, keys above it, keys in it
    __shared__ unsigned n_out;
    unsigned long long prefix = 0ull, mask = 0ull;
    int need = k;
    for (int shift = 56; shift >= 0; shift -= 8) {
        if (shift == 40) {
            const unsigned hi = (unsigned)(prefix >> 48);
            prefix |= (hi != 0 && !(hi & 0x8000u)) ? 0xffffull << 32 : 0ull;
            mask |= 0xffffull << 32;
            shift = 24;
        }
        hist[threadIdx.x] = 0u;   // 256 threads
        __syncthreads();
#pragma unroll
        for (int i = 0; i < KPT; i++)
            if ((key[i] & mask) == prefix) atomicAdd(&hist[(key[i] >> shift) & 255], 1u);
        __syncthreads();
        if (threadIdx.x < 64) {   // lane l holds the bins 255 - 4 l .. 252 - 4 l: counts above them by a scan over the lanes
            const int l = threadIdx.x;
            unsigned c[4], own = 0u;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                c[j] = hist[255 - 4 * l - j];
                own += c[j];
            }
            unsigned upto = own;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const unsigned t = __shfl_up(upto, o, 64);
                if (l >= o) upto += t;
            }
            unsigned above = upto - own;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (above < (unsigned)need && above + c[j] >= (unsigned)need) {   // one bin of one lane
                    pick[0] = (unsigned)(255 - 4 * l - j);
                    pick[1] = above;
                    pick[2] = c[j];
                }
                above += c[j];
            }
        }
        __syncthreads();
        prefix |= (unsigned long long)pick[0] << shift;
        mask |= 255ull << shift;
        need -= (int)pick[1];
        const bool done = pick[2] == (unsigned)need;
        __syncthreads();
        if (done) break;   // block-uniform
    }
    if (threadIdx.x == 0) n_out = 0u;
    for (int i = threadIdx.x; i < k; i += 256) out[i] = 0ull;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < KPT; i++)
        if (key[i] != 0ull && (key[i] & mask) >= prefix) out[atomicAdd(&n_out, 1u)] = key[i];
    __syncthreads();
}

// How many of keys[0, n) (LDS; a zero behind them where n is odd) are above `own`: its place among them in descending order, the
// keys being distinct.  Two keys a read that serves the whole wave, no barriers: 0.5 us for 50 keys, where a bitonic sort of 64 in
// LDS took 21 barriers, 4 us.
__device__ __forceinline__ int rank_of(unsigned long long own, const unsigned long long* keys, int n) {
    const ulonglong2* two = reinterpret_cast<const ulonglong2*>(keys);
    int above = 0;
#pragma unroll 8
    for (int j = 0; j < (n + 1) / 2; j++) {
        const ulonglong2 q = two[j];
        above += (q.x > own) + (q.y > own);
    }
    return above;
}

// The k best of a slice, in descending order, zeros behind the last.
__global__ __launch_bounds__(256) void topk_slice_kernel(const uint16_t* __restrict__ logits, int64_t V,
                                                         int64_t ld, int k,
                                                         unsigned long long* __restrict__ cand) {
    constexpr int KPT = kSlice / 256;
    const int64_t m = blockIdx.y;
    const int64_t base = (int64_t)blockIdx.x * kSlice;
    const uint16_t* row = logits + m * ld;
    unsigned long long key[KPT];
    uint16_t v[KPT];
#pragma unroll
    for (int i = 0; i < KPT; i++) {
        const int64_t idx = base + threadIdx.x + 256 * i;
        v[i] = row[idx < V ? idx : V - 1];
    }
#pragma unroll
    for (int i = 0; i < KPT; i++) {
        const int64_t idx = base + threadIdx.x + 256 * i;
        key[i] = idx < V ? sel_key(bf2f(v[i]), (uint32_t)idx) : 0ull;
    }
    __shared__ __attribute__((aligned(16))) unsigned long long top[kMaxTopK + 2];
    if (threadIdx.x == 0) top[k] = 0ull;
    radix_top<KPT>(key, k, top);   // (at least k keys: k <= kMaxTopK <= kSlice; ends in a barrier)
    const int i = threadIdx.x;
    if (i >= k) return;
    const unsigned long long own = top[i];   // (zeros stand behind the keys)
    cand[(m * gridDim.x + blockIdx.x) * (int64_t)k + (own != 0ull ? rank_of(own, top, k) : i)] = own;
}

// cuRAND XORWOW, curand_init(seed, subsequence = 0, offset = 0) (no skip-ahead)
// and curand_uniform — restated from the published curand_kernel.h.
__device__ __forceinline__ float xorwow_uniform_first(uint64_t seed) {
    uint32_t s0 = (uint32_t)seed ^ 0xaad26b49u;
    uint32_t s1 = (uint32_t)(seed >> 32) ^ 0xf7dcefddu;
    uint32_t t0 = 1099087573u * s0;
    uint32_t t1 = 2591861531u * s1;
    uint32_t d = 6615241u + t1 + t0;
    uint32_t v0 = 123456789u + t0, v4 = 5783321u + t0;
    uint32_t t = v0 ^ (v0 >> 2);
    uint32_t nv4 = (v4 ^ (v4 << 4)) ^ (t ^ (t << 1));
    d += 362437u;
    uint32_t x = nv4 + d;
    return x * 2.3283064e-10f + (2.3283064e-10f / 2.0f);
}

// One block per row: the k best of the slices' candidates, sorted, then temperature, softmax and one draw
// (logit_decode.cu:225-272) by one wave that holds candidate i in lane i % 64: the exponentials side by side, the sums in the
// reference's order.
// Bound by its steps' latencies.  Of `full` whole slices the least key in place ceil(k / full) has k keys at or above it, so what is
// below it is left out first: of 151,936 logits and k = 50 some 250 of 1,900 candidates stay and are put in order at once, where a
// radix selection makes four to six passes of 1.5 us.  It is still made where more than kFew stay (a few slices with all the best).
// The running sums are made once: the total, the nucleus and the draw read them (were four chains of k additions).  us of a
// call with its slices, 7 rows of 151,936 logits, k = 50: 30 to 35 -> 25; k = 256: 58 to 100 -> 42 to 56.
constexpr int kFew = 768;
template <int KPT>
__global__ __launch_bounds__(256) void topk_merge_sample_kernel(const unsigned long long* __restrict__ cand,
                                                                int nb, int full, int k, float temperature,
                                                                float top_p, uint64_t seed,
                                                                const int32_t* step, int32_t* ids) {
#pragma clang fp contract(off)
    __shared__ unsigned long long sk[kMaxTopK];
    __shared__ __attribute__((aligned(16))) unsigned long long few[kFew];
    __shared__ int n_few;
    const int64_t m = blockIdx.x;
    const int total = nb * k, lane = threadIdx.x & 63;
    unsigned long long key[KPT];
#pragma unroll
    for (int i = 0; i < KPT; i++) {
        const int j = threadIdx.x + 256 * i;
        const unsigned long long c = cand[m * total + (j < total ? j : total - 1)];
        key[i] = j < total ? c : 0ull;
    }
    sk[threadIdx.x] = 0ull;
    for (int i = threadIdx.x; i < kFew; i += 256) few[i] = 0ull;
    if (threadIdx.x == 0) n_few = 0;
    unsigned long long least = 0ull;   // complemented: the maximum's
    if (full > 0) {
        const int at = (k + full - 1) / full - 1;
        for (int q = lane; q < full; q += 64) {
            const unsigned long long c = ~cand[m * total + (int64_t)q * k + at];
            least = c > least ? c : least;
        }
        least = ~wave_max(least);
    }
    __syncthreads();
    int mine = 0;   // the wave's
#pragma unroll
    for (int i = 0; i < KPT; i++) mine += __popcll(__ballot(key[i] != 0ull && key[i] >= least));
    int at = 0;
    if (lane == 0) at = atomicAdd(&n_few, mine);
    at = __builtin_amdgcn_readfirstlane(at);
#pragma unroll
    for (int i = 0; i < KPT; i++) {
        const bool in = key[i] != 0ull && key[i] >= least;
        const unsigned long long who = __ballot(in);
        const int to = at + __popcll(who & ((1ull << lane) - 1ull));
        if (in && to < kFew) few[to] = key[i];
        at += __popcll(who);
    }
    __syncthreads();
    int n_in = n_few;
    if (n_in > kFew) {   // block-uniform
        radix_top<KPT>(key, k, few);
        if (threadIdx.x == 0) few[k] = 0ull;   // (k <= kMaxTopK < kFew)
        n_in = k;
        __syncthreads();
    }
    for (int i = threadIdx.x; i < n_in; i += 256) {
        const unsigned long long own = few[i];
        const int to = rank_of(own, few, n_in);
        if (own != 0ull && to < k) sk[to] = own;
    }
    __syncthreads();
    if (threadIdx.x >= 64) return;
    constexpr int J = kMaxTopK / 64;
    int n = 0;
    float e[J];
    const float T = temperature > 0.0f ? temperature : 1.0f;
    const float max_val = key_val(sk[0]) / T;   // the keys are sorted by value
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int i = 64 * j + lane;
        const unsigned long long c = i < k ? sk[i] : 0ull;
        n += __popcll(__ballot(c != 0ull));
        e[j] = c != 0ull ? expf(key_val(c) / T - max_val) : 0.f;
    }
    if (n == 0) {
        if (lane == 0) ids[m] = -1;
        return;
    }
    float upto[J], c = 0.0f;   // sums of the weights up to a candidate's, in order
#pragma unroll
    for (int j = 0; j < J; j++) {
        upto[j] = 0.0f;
#pragma unroll 8
        for (int l = 0; l < min(64, n - 64 * j); l++) {
            c += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, e[j]), l));
            if (lane == l) upto[j] = c;
        }
    }
    auto sum_to = [&](int i) {   // i uniform
        float v = upto[0];
#pragma unroll
        for (int j = 1; j < J; j++) v = i >= 64 * j ? upto[j] : v;
        return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), i & 63));
    };
    auto first = [&](auto holds, int none) {   // the first of n candidates whose running sum holds
        int f = none;
#pragma unroll
        for (int j = J - 1; j >= 0; j--) {
            const unsigned long long b = __ballot(64 * j + lane < n && holds(upto[j]));
            if (b) f = 64 * j + __ffsll(b) - 1;
        }
        return f;
    };
    float sum = sum_to(n - 1);
    if (top_p > 0.0f && top_p < 1.0f) {
        n = first([&](float s) { return s >= top_p * sum; }, n - 1) + 1;
        sum = sum_to(n - 1);
    }
    const uint64_t sd = seed + (step ? (uint64_t)(int64_t)step[m] : 0ull);
    const float u = xorwow_uniform_first(sd) * sum;
    const int picked = first([&](float s) { return u <= s; }, n - 1);
    if (lane == 0) ids[m] = key_idx(sk[picked]);
}

}  // namespace qie

using namespace qie;

extern "C" {

int64_t qie_sample_workspace_bytes(int64_t M, int64_t V) {
    const int64_t nb = (V + kSlice - 1) / kSlice;
    return M * nb * kMaxTopK * 8 + M * 8 + 64;
}

int qie_keys_to_ids(const uint64_t* keys, int64_t M, int32_t* out_ids, void* stream) {
    QIE_REQUIRE(keys && out_ids && M >= 0, "qie_keys_to_ids: bad arguments");
    if (M == 0) return 0;
    hipLaunchKernelGGL(keys_to_ids_kernel, dim3((unsigned)((M + 63) / 64)), dim3(64), 0,
                       (hipStream_t)stream, (const unsigned long long*)keys, M, out_ids);
    QIE_LAUNCH_CHECK();
    return 0;
}

int qie_sample(const void* logits, int64_t M, int64_t V, int64_t ld, const qie_sampling* s,
               const int32_t* step_dev, int32_t* out_ids, void* ws, void* stream) {
    QIE_REQUIRE(logits && s && out_ids && ws && M >= 0 && V > 0 && V < (1 << 24) && ld >= V,
                "qie_sample: bad arguments");
    if (M == 0) return 0;
    hipStream_t st = (hipStream_t)stream;
    if (s->top_k <= 1) {
        unsigned long long* keys = (unsigned long long*)ws;
        QIE_HIP(hipMemsetAsync(keys, 0, M * 8, st));
        hipLaunchKernelGGL(argmax_keys_kernel, dim3(64, (unsigned)M), dim3(256), 0, st,
                           (const uint16_t*)logits, V, ld, keys);
        QIE_LAUNCH_CHECK();
        return qie_keys_to_ids((const uint64_t*)keys, M, out_ids, stream);
    }
    int k = s->top_k;
    if (k > V) k = (int)V;
    if (k > kMaxTopK) k = kMaxTopK;
    const int nb = (int)((V + kSlice - 1) / kSlice);
    unsigned long long* cand = (unsigned long long*)ws;
    hipLaunchKernelGGL(topk_slice_kernel, dim3(nb, (unsigned)M), dim3(256), 0, st,
                       (const uint16_t*)logits, V, ld, k, cand);
    QIE_LAUNCH_CHECK();
    const int total = nb * k;
    // a thread of the merge holds up to 64 candidates in registers
    QIE_REQUIRE(total <= 64 * 256, "qie_sample: top-k of %d over %lld logits leaves %d candidates, more than %d", k, (long long)V, total, 64 * 256);
    const auto fn = total <= 8 * 256 ? topk_merge_sample_kernel<8> : total <= 40 * 256 ? topk_merge_sample_kernel<40>
                                                                                       : topk_merge_sample_kernel<64>;
    hipLaunchKernelGGL(fn, dim3((unsigned)M), dim3(256), 0, st, cand, nb, (int)(V / kSlice), k,
                       s->temperature, s->top_p, (uint64_t)s->seed, step_dev, out_ids);
    QIE_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
