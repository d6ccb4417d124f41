// k_gemv_row.hip — one-row projections on bf16 weights whose rows are few enough for all of them to be in flight at once.
//
//   y[N] = x[K] . W[N, K]^T (RMSNorm of x in front where asked for; STORE, RESIDUAL, F32), K <= 5,120, N <= 32 rows a CU
//
// Such a launch lasts two trips to memory: x (and the norm), and the weights, which need every CU and every byte asked for
// early.  k_gemv.hip gives a wave two rows, U chunks of them at a time, then the next two: Qwen2-0.5B's down projection (896 rows of
// 4,864) ran on 112 blocks in two chunks, Qwen3-14B's O and QKV in rounds.  Here a wave owns one row and holds all of it in
// registers (U 16-byte pieces a lane, asked for before anything is computed), and the blocks' sizes spread the rows evenly over
// the CUs.  us a launch inside the decode, before -> now: Qwen2-0.5B down 6.3 -> 3.5, QKV 4.0 -> 3.0, O 3.4 -> 3.0; Qwen2-7B QKV
// 9.6 -> 8.2, O 6.9 -> 6.0; Qwen3-14B QKV 17.0 -> 14.6, O 12.1 -> 9.8.
// (SwiGLU with the gate and up row in one wave, measured and dropped: Qwen2-0.5B 5.8 -> 6.3 to 7.3; its rows come several a wave
// and the norm is paid once a wave's life in k_gemv.hip.)
#include "qie_common.hpp"
#include "../../include/qie/qie_ops.h"

#include <algorithm>
#include <type_traits>

namespace qie {

typedef unsigned int gr_u32x4 __attribute__((ext_vector_type(4)));

struct GemvRowParams {
    const uint16_t* x;
    const uint16_t* norm_w;
    float eps;
    int numerics;
    const uint16_t* w[3];
    const uint16_t* bias[3];
    int n0, n01;   // rows of segment 0, of segments 0 and 1
    int K, N;
    uint16_t* y;
};

// XV: pieces of x a thread stages (64 U <= XV threads)
template <int EPI, int U, int XV, bool NORM>
__global__ __launch_bounds__(1024) void gemv_row_kernel(GemvRowParams p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    gr_u32x4* xs = reinterpret_cast<gr_u32x4*>(smem);
    float* red = reinterpret_cast<float*>(smem + U * 1024);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int NW = blockDim.x >> 6, T = blockDim.x, K = p.K;
    const int out = (int)blockIdx.x * NW + wave, col = out < p.N ? out : p.N - 1;   // waves past N: the last row again
    auto rsrc = [](const void* base, int64_t bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
    };
    // x first: vmcnt retires in order.  A piece past K reads zeros (range check), without a branch.
    const auto rx = rsrc(p.x, (int64_t)K * 2), rn = rsrc(NORM ? p.norm_w : p.x, (int64_t)K * 2);
    gr_u32x4 xv[XV], nv[NORM ? XV : 1];
#pragma unroll
    for (int v = 0; v < XV; v++) {
        xv[v] = __builtin_amdgcn_raw_buffer_load_b128(rx, (tid + v * T) * 16, 0, 0);
        if constexpr (NORM) nv[v] = __builtin_amdgcn_raw_buffer_load_b128(rn, (tid + v * T) * 16, 0, 0);
    }
    // the epilogue's operand: the old value, or the bias (none: element 0 of x, unused)
    const uint16_t* bias = nullptr;
    uint32_t ep = 0;
    if constexpr (EPI == QIE_EPI_RESIDUAL) {
        ep = __builtin_amdgcn_raw_buffer_load_b16(rsrc(p.y, (int64_t)p.N * 2), col * 2, 0, 0);
    } else if constexpr (EPI == QIE_EPI_STORE) {
        bias = col < p.n0 ? p.bias[0] : (col < p.n01 ? p.bias[1] : p.bias[2]);
        const int bi = col < p.n0 ? col : (col < p.n01 ? col - p.n0 : col - p.n01);
        ep = __builtin_amdgcn_raw_buffer_load_b16(rsrc(bias ? bias : p.x, bias ? (int64_t)(bi + 1) * 2 : 2), bias ? bi * 2 : 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    const uint16_t* base = col < p.n0    ? p.w[0] + (int64_t)col * K
                           : col < p.n01 ? p.w[1] + (int64_t)(col - p.n0) * K
                                         : p.w[2] + (int64_t)(col - p.n01) * K;
    const auto rw = rsrc(base, (int64_t)K * 2);
    gr_u32x4 wv[U];
#pragma unroll
    for (int u = 0; u < U; u++) wv[u] = __builtin_amdgcn_raw_buffer_load_b128(rw, lane * 16, u * 1024, 2);   // nt: read once
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int v = 0; v < XV; v++) {   // x's arithmetic stays behind the weights' issue
        asm volatile("" : "+v"(xv[v]));
        if constexpr (NORM) asm volatile("" : "+v"(nv[v]));
    }
    auto put = [&]() {   // the thread's pieces -> LDS (pieces past K: zeros)
#pragma unroll
        for (int v = 0; v < XV; v++)
            if (tid + v * T < 64 * U) xs[tid + v * T] = xv[v];
    };
    auto meet = [&]() {   // (not __syncthreads: the weights stay in flight)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (NORM) {
        // The sum of squares is taken by the first four waves in the order of a block of 256 threads, whatever this block's
        // size: the persistent decode step (k_persist.hip) gives the same bits.
        constexpr int XS = (U * 64 + 255) / 256;
        put();
        meet();
        if (wave < 4) {
            float ss = 0.f;
#pragma unroll
            for (int c = 0; c < XS; c++) {
                if (wave * 64 + c * 256 >= 64 * U) break;   // wave-uniform: the image ends
                const gr_u32x4 s = xs[tid + c * 256];
                const uint32_t e[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float a = bf_lo(e[j]), b = bf_hi(e[j]);
                    ss += a * a;
                    ss += b * b;
                }
            }
            ss = wave_sum(ss);
            if (lane == 0) red[wave] = ss;
        }
        meet();
        float tot = 0.f;
        for (int w = 0; w < 4; w++) tot += red[w];
        const float rms = sqrtf((tot / (float)K) + p.eps), inv = 1.0f / rms;
        auto apply = [&](auto hf) {
            constexpr bool HF = decltype(hf)::value;
#pragma unroll
            for (int v = 0; v < XV; v++) {
#pragma clang fp contract(off)
                if (wave * 64 + v * T >= 64 * U) break;   // wave-uniform: no piece
                uint32_t e[4] = {xv[v].x, xv[v].y, xv[v].z, xv[v].w};
                const uint32_t w[4] = {nv[v].x, nv[v].y, nv[v].z, nv[v].w};
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    if (HF) e[j] = pack2(bf_lo(w[j]) * rbf(bf_lo(e[j]) * inv), bf_hi(w[j]) * rbf(bf_hi(e[j]) * inv));
                    else e[j] = pack2((bf_lo(e[j]) / rms) * bf_lo(w[j]), (bf_hi(e[j]) / rms) * bf_hi(w[j]));
                }
                xv[v] = gr_u32x4{e[0], e[1], e[2], e[3]};
            }
        };
        if (p.numerics == QIE_NUMERICS_HF) apply(std::true_type{});
        else apply(std::false_type{});
    }
    put();
    meet();
    float acc = 0.f;
#pragma unroll
    for (int u = 0; u < U; u++) {
        const gr_u32x4 xq = xs[u * 64 + lane];
        const uint32_t e[4] = {xq.x, xq.y, xq.z, xq.w}, f[4] = {wv[u].x, wv[u].y, wv[u].z, wv[u].w};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            acc = fmaf(bf_lo(e[j]), bf_lo(f[j]), acc);
            acc = fmaf(bf_hi(e[j]), bf_hi(f[j]), acc);
        }
    }
    acc = wave_sum(acc);
    if (lane != 0 || out >= p.N) return;
    if constexpr (EPI == QIE_EPI_F32) reinterpret_cast<float*>(p.y)[out] = acc;
    else if constexpr (EPI == QIE_EPI_RESIDUAL) p.y[out] = f2bf(bf2f((uint16_t)ep) + rbf(acc));
    else p.y[out] = f2bf(bias ? acc + bf2f((uint16_t)ep) : acc);
}

namespace {
template <int EPI, int U>
void gr_launch_u(const GemvRowParams& p, unsigned grid, unsigned threads, hipStream_t st) {
    const size_t lds = (size_t)U * 1024 + 64;
    const bool one = 64 * U <= (int)threads;
    auto k = p.norm_w ? (one ? gemv_row_kernel<EPI, U, 1, true> : gemv_row_kernel<EPI, U, 3, true>)
                      : (one ? gemv_row_kernel<EPI, U, 1, false> : gemv_row_kernel<EPI, U, 3, false>);
    hipLaunchKernelGGL(k, dim3(grid), dim3(threads), lds, st, p);
}
template <int EPI>
void gr_launch(const GemvRowParams& p, int u, unsigned grid, unsigned threads, hipStream_t st) {
    if (u == 2) return gr_launch_u<EPI, 2>(p, grid, threads, st);
    if (u == 4) return gr_launch_u<EPI, 4>(p, grid, threads, st);
    if (u == 7) return gr_launch_u<EPI, 7>(p, grid, threads, st);
    gr_launch_u<EPI, 10>(p, grid, threads, st);
}
}  // namespace

// *done false: not its shape
int gemv_row(const qie_linear_args* a, hipStream_t st, bool* done) {
    const int64_t cus = device_cu_count(), per_cu = (a->N + cus - 1) / cus;
    *done = a->M == 1 && !(a->flags & QIE_LINEAR_FP8) && a->epilogue != QIE_EPI_SWIGLU && !a->argmax_keys && a->K <= 5120 &&
            per_cu <= 32 && ((uintptr_t)a->norm_w) % 16 == 0;   // 32 waves a CU: 64 registers, the largest form's
    if (!*done) return 0;
    GemvRowParams p{};
    p.x = (const uint16_t*)a->x;
    p.norm_w = (const uint16_t*)a->norm_w;
    p.eps = a->norm_eps;
    p.numerics = a->numerics;
    for (int i = 0; i < 3; i++) {
        p.w[i] = (const uint16_t*)a->w[i];
        p.bias[i] = (const uint16_t*)a->bias[i];
    }
    p.n0 = (int)a->seg_rows[0];
    p.n01 = (int)(a->seg_rows[0] + a->seg_rows[1]);
    p.K = (int)a->K;
    p.N = (int)a->N;
    p.y = (uint16_t*)a->y;
    const int u = a->K <= 1024 ? 2 : a->K <= 2048 ? 4 : a->K <= 3584 ? 7 : 10;
    // Waves a block: a CU's rows in whole blocks.  With the norm as few blocks as can be (every block norms x; 7B QKV, 18 rows a CU:
    // two of 9 waves 8.2 us, three of 6 9.3; 14B QKV, 28 rows: two of 14 14.6, four of 7 16.1), else 4 waves or the next size up to
    // 8 that divides the rows better (7B O, 14 rows: one of 14 waves 6.5 us, two of 7 6.0, three and a half of 4 6.3; 14B O, 20 rows:
    // two of 10 10.3, four of 5 11.0, five of 4 9.8).
    int64_t nw;
    if (a->norm_w) {
        const int64_t blocks = (per_cu + 15) / 16;
        nw = std::max<int64_t>(4, (per_cu + blocks - 1) / blocks);
    } else {
        nw = 4;
        auto rounded = [&](int64_t w) { return (per_cu + w - 1) / w * w; };
        for (int64_t w = 5; w <= 8; w++)
            if (rounded(w) < rounded(nw)) nw = w;
    }
    const unsigned grid = (unsigned)((a->N + nw - 1) / nw), threads = (unsigned)(64 * nw);
    switch (a->epilogue) {
        case QIE_EPI_RESIDUAL: gr_launch<QIE_EPI_RESIDUAL>(p, u, grid, threads, st); break;
        case QIE_EPI_F32: gr_launch<QIE_EPI_F32>(p, u, grid, threads, st); break;
        default: gr_launch<QIE_EPI_STORE>(p, u, grid, threads, st);
    }
    QIE_LAUNCH_CHECK();
    return 0;
}

}  // namespace qie
