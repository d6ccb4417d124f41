// k_gemm_mid.hip — MFMA bf16 GEMM for prompts of a few dozen to about a thousand rows.
//
//   C[M, N] = A[M, K] . W[N, K]^T, fp32 accumulation, the epilogues of k_gemm.hip.
//
// At these row counts the weights come from HBM once and the 256x256 tiles of the long-prompt kernels leave most of the
// chip idle (Qwen2-7B, 301 rows: 2 x 14 tiles for the O and down projections), while the register-staged 128x128 kernel
// holds one k-tile in flight and waits a memory round trip (about 1 us) for every 64 of K.  Here:
//   * a BM x BN tile (64x64 to 320x160), BK = 64, in a ring of LDS slots filled by LDS-DMA: all slots but one are in flight,
//     one barrier per k-tile;
//   * what bounds it: one CU fills its LDS at 130-140 GB/s with lines of its L2, 97 of the Infinity Cache, 54-64 of HBM (some 40 KB of
//     requests in flight at their latency; rings of 2 to 9 slots, split roles of waves and prefetches into L2 by the same CUs all
//     measured the same), so the time follows the rows of A and W that a CU stages for its outputs: tall tiles, and columns in tiles
//     that fill rounds of the chip.  Qwen2-7B gate / up, 128 / 160 columns a tile: 113 rows 71 / 58 us, 200 rows 97 / 78, 301 rows 120 /
//     97, 512 rows 171 / 143;
//   * 8 waves as 2 (M) x 2 (N) x 2 (K halves of every k-tile): a wave's tile is half the block's in both directions, which
//     reads LDS as often as four waves would, and two waves a SIMD cover each other's fragment reads.  The K halves meet in
//     LDS once, behind the loop;
//   * split-K over workgroups where the tiles do not fill the chip (fp32 slabs, the last arriver sums them in part order:
//     gemm8_kernel's protocol, the result does not depend on arrival order);
//   * workgroups that share a weight tile are neighbours in one XCD, parts are the slowest index: an XCD's L2 holds one K
//     range of A.
#include "gemm_impl.hpp"
#include "gemm_plan.hpp"

#include <algorithm>

namespace qie {

// weight row of tile column c of column tile nt.  SwiGLU: a lane of the epilogue holds columns 4 g .. 4 g + 3 of every fragment, so
// those are two gate rows and the same outputs' up rows; two fragments give it four outputs side by side (a last odd one two)
template <int EPI, int BN>
__device__ __forceinline__ const uint16_t* mid_wrow(const GemmParams& p, int64_t nt, int c) {
    if constexpr (EPI == QIE_EPI_SWIGLU) {
        constexpr int TN = BN / 2, FJ = TN / 16;
        const int cs = c % TN, f = cs / 16, g = (cs % 16) / 4, r = cs % 4;
        const int jl = f / 2 * 16 + (f == FJ - 1 && FJ % 2 ? 2 * g : 4 * g + 2 * (f % 2)) + (r & 1);
        const int64_t j = nt * TN + (c / TN) * (TN / 2) + jl;
        const int64_t jj = j < p.N ? j : p.N - 1;
        return (r >= 2 ? p.w1 : p.w0) + jj * p.K;
    } else {
        const int64_t r = nt * BN + c;
        const int64_t rr = r < p.N ? r : p.N - 1;
        if (rr < p.n0) return p.w0 + rr * p.K;
        if (rr < p.n01) return p.w1 + (rr - p.n0) * p.K;
        return p.w2 + (rr - p.n01) * p.K;
    }
}

template <int EPI, int BM, int BN, int SLOTS>
__global__ __launch_bounds__(512) void gemm_mid_kernel(GemmParams p, int n_mt, int n_nt, int gm, int whole, G8Split sk, TailOf<EPI> tail) {
#pragma clang fp contract(off)
    constexpr int TM = BM / 2, TN = BN / 2, FI = TM / 16, FJ = TN / 16, FH = FI / 2;
    constexpr int SLOT = (BM + BN) * 128;      // A rows, then W rows, 128 B each
    // LDS-DMA instructions (8 rows each) per wave and k-tile; where the waves don't share them evenly, the first MORE have one more
    constexpr int BLOCKS = (BM + BN) / 8, IPW = (BLOCKS + 7) / 8, MORE = BLOCKS % 8;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;
    const int fr = lane & 15, g = lane >> 4;
    // workgroups [0, whole): a tile each; behind them the other tiles, splitk parts each.  Within either range the
    // bijective XCD remap keeps neighbours (the M tiles of a weight tile) on one XCD
    const bool cut = (int)blockIdx.x >= whole;
    const int nwg = cut ? gridDim.x - whole : whole, orig = cut ? blockIdx.x - whole : blockIdx.x;
    const int q8 = nwg >> 3, r8 = nwg & 7, xcd = orig & 7;
    const int wid = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + (orig >> 3);
    const int parts = cut ? sk.splitk : 1, cuts = quotient(nwg, parts);   // cut tiles: part-major, so an XCD's parts share a K range of A
    const int part = quotient(wid, cuts), ct = wid - part * cuts, tile = cut ? whole + ct : wid;
    int mti, nti;
    banded(tile, n_mt, n_nt, gm, &mti, &nti);
    const int64_t mt = mti, nt = nti, m0 = mt * BM;

    const int nk_all = (int)(p.K / mid::BK);
    const int kb = (int)((int64_t)part * nk_all / parts);        // this part's k-tiles [kb, kb + nk)
    const int nk = (int)((int64_t)(part + 1) * nk_all / parts) - kb;

    // instruction i of this wave fills the slot's rows 8 b .. 8 b + 7, b = 8 i + wave: lane -> row 8 b + (lane >> 3),
    // LDS chunk lane & 7, which holds the source's chunk (lane & 7) ^ swz(row)
    const uint16_t* src[IPW];
#pragma unroll
    for (int i = 0; i < IPW; i++) {
        if (MORE && i == IPW - 1 && wave >= MORE) break;   // uniform
        const int r = 8 * (8 * i + wave) + (lane >> 3);
        const int cs = (lane & 7) ^ g8_swz(r);
        if (r < BM) {   // uniform over the wave: BM is a multiple of 8
            int64_t ar = m0 + r;
            ar = ar < p.M ? ar : p.M - 1;   // rows past M: re-read row M - 1, never stored
            src[i] = p.A + ar * p.lda + (int64_t)kb * mid::BK + cs * 8;
        } else {
            src[i] = mid_wrow<EPI, BN>(p, nt, r - BM) + (int64_t)kb * mid::BK + cs * 8;
        }
    }
    // kEpiQkv of small tiles: its operands are on their way before the first k-tile
    constexpr bool EARLY = EPI == kEpiQkv && FH * FJ <= 8;
    [[maybe_unused]] QkvOps<FH> ops[EARLY ? FJ : 1];
    if constexpr (EARLY) {
#pragma unroll
        for (int j = 0; j < FJ; j++) qkv_load(p, tail, m0 + wm * TM + wk * (FH * 16) + fr, nt * BN + wn * TN + 16 * j + 4 * g, ops[j]);
        __builtin_amdgcn_sched_barrier(0);
    }
    auto stage = [&](int kt, int slot) {
        unsigned char* dst = smem + slot * SLOT + wave * 1024;
#pragma unroll
        for (int i = 0; i < IPW; i++) {
            if (MORE && i == IPW - 1 && wave >= MORE) break;
            glds16(src[i] + (int64_t)kt * mid::BK, dst + i * 8192);
        }
    };

    f32x4 acc[FI][FJ];
#pragma unroll
    for (int i = 0; i < FI; i++)
#pragma unroll
        for (int j = 0; j < FJ; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int t = 0; t < SLOTS - 1 && t < nk; t++) stage(t, t);
    int slot = 0, fill = SLOTS - 1;
    for (int t = 0; t < nk; t++) {
        // k-tile t has landed (the SLOTS - 2 younger ones may still fly), and every wave is done with the slot of t - 1
        if (t + SLOTS - 1 <= nk && (MORE == 0 || wave < MORE)) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(IPW * (SLOTS - 2)) : "memory");
        else if (t + SLOTS - 1 <= nk) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((IPW - 1) * (SLOTS - 2)) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (t + SLOTS - 1 < nk) stage(t + SLOTS - 1, fill);
        const unsigned char* buf = smem + slot * SLOT;
        bf16x8 fa[FI], fb[FJ];
        auto read_a = [&](int i) {
            const int row = wm * TM + i * 16 + fr;
            fa[i] = *reinterpret_cast<const bf16x8*>(buf + row * 128 + (((4 * wk + g) ^ g8_swz(row)) * 16));
        };
#pragma unroll
        for (int j = 0; j < FJ; j++) {
            const int row = BM + wn * TN + j * 16 + fr;
            fb[j] = *reinterpret_cast<const bf16x8*>(buf + row * 128 + (((4 * wk + g) ^ g8_swz(row)) * 16));
        }
        constexpr int AHEAD = BM >= 256 ? 2 : FI;   // tall tiles: two A fragments on their way while one is multiplied
#pragma unroll
        for (int i = 0; i < AHEAD; i++) read_a(i);
#pragma unroll
        for (int i = 0; i < FI; i++) {
            if (i + AHEAD < FI) read_a(i + AHEAD);
            if (AHEAD < FI) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < FJ; j++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0);   // W Aᵀ
            if (AHEAD < FI) __builtin_amdgcn_sched_barrier(0);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // this wave's reads of the slot are done
        __builtin_amdgcn_sched_barrier(0);
        slot = slot + 1 == SLOTS ? 0 : slot + 1;
        fill = fill + 1 == SLOTS ? 0 : fill + 1;
    }

    // ---------------- the two K halves: wave w and w ^ 4 hold the same tile; each keeps half of its rows
    f32x4 res[FH][FJ];
    {
        f32x4* ex = reinterpret_cast<f32x4*>(smem);
        constexpr int FIT = SLOTS * SLOT / (8 * FH * 1024), JN = FIT < FJ ? FIT : FJ;   // fragment columns the LDS takes at once
        static_assert(JN >= 1, "exchange area");
#pragma unroll
        for (int j0 = 0; j0 < FJ; j0 += JN) {
            __syncthreads();
#pragma unroll
            for (int i = 0; i < FH; i++)
#pragma unroll
                for (int j = j0; j < j0 + JN && j < FJ; j++) {
                    if (wk == 0) {
                        ex[((wave * FH + i) * JN + j - j0) * 64 + lane] = acc[FH + i][j];
                        res[i][j] = acc[i][j];
                    } else {
                        ex[((wave * FH + i) * JN + j - j0) * 64 + lane] = acc[i][j];
                        res[i][j] = acc[FH + i][j];
                    }
                }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < FH; i++)
#pragma unroll
                for (int j = j0; j < j0 + JN && j < FJ; j++) res[i][j] = res[i][j] + ex[(((wave ^ 4) * FH + i) * JN + j - j0) * 64 + lane];
        }
    }

    if (parts > 1) {   // uniform
        constexpr int SLAB = BM * BN;   // floats
        const int64_t tb = (int64_t)ct * parts;
        const auto rs = __builtin_amdgcn_make_buffer_rsrc(sk.slab + (tb + part) * SLAB, (short)0, SLAB * 4, 0x00020000);
#pragma unroll
        for (int i = 0; i < FH; i++)
#pragma unroll
            for (int j = 0; j < FJ; j++)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_g8, res[i][j]), rs,
                                                       (((wave * FH + i) * FJ + j) * 64 + lane) * 16, 0, 16);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // every storing wave drains
        __syncthreads();
        int* flag = reinterpret_cast<int*>(smem);
        if (tid == 0) {
            const unsigned old = __hip_atomic_fetch_add(sk.cnt + ct, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *flag = old == (unsigned)parts - 1 ? 1 : 0;
        }
        __syncthreads();
        if (*flag == 0) return;   // uniform
        // part order: independent of who arrived last; QN parts' loads in flight (one after the other cost 0.75 us each)
        constexpr int QN = FH * FJ >= 16 ? 1 : 16 / (FH * FJ);
        for (int q0 = 0; q0 < parts; q0 += QN) {
            f32x4 v[QN][FH][FJ];
#pragma unroll
            for (int u = 0; u < QN; u++) {
                const int q = q0 + u < parts ? q0 + u : parts - 1;
                const auto rq = __builtin_amdgcn_make_buffer_rsrc(sk.slab + (tb + q) * SLAB, (short)0, SLAB * 4, 0x00020000);
#pragma unroll
                for (int i = 0; i < FH; i++)
#pragma unroll
                    for (int j = 0; j < FJ; j++)
                        v[u][i][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                                   rq, (((wave * FH + i) * FJ + j) * 64 + lane) * 16, 0, 16));
            }
#pragma unroll
            for (int u = 0; u < QN; u++) {
                if (q0 + u >= parts) break;
#pragma unroll
                for (int i = 0; i < FH; i++)
#pragma unroll
                    for (int j = 0; j < FJ; j++) res[i][j] = q0 + u == 0 ? v[u][i][j] : res[i][j] + v[u][i][j];
            }
        }
        if (tid == 0) __hip_atomic_store(sk.cnt + ct, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // ---------------- epilogue.  D = W Aᵀ: a lane holds row m = lane & 15 and the columns 4 g .. 4 g + 3 of a fragment, one
    // 8- (fp32: 16-) byte store where C's rows allow it
    const bool vec = p.vec != 0;
    const int64_t row0 = m0 + wm * TM + wk * (FH * 16) + fr;
    if constexpr (EPI == QIE_EPI_SWIGLU) {
#pragma unroll
        for (int m = 0; m < (FJ + 1) / 2; m++) {
            constexpr int PAIRS = FJ / 2;
            const int n = m < PAIRS ? 4 : 2;   // outputs
            const int64_t col = nt * TN + (TN / 2) * wn + 16 * m + n * g;
#pragma unroll
            for (int i = 0; i < FH; i++) {
                const int64_t row = row0 + i * 16;
                if (row >= p.M) continue;
                float h[4];
#pragma unroll
                for (int r = 0; r < n; r++) {
                    const f32x4 v = res[i][2 * m + r / 2];
                    const float gg = rbf(v[r & 1]);
                    const float uu = rbf(v[2 + (r & 1)]);
                    h[r] = uu * rbf(gg * (1.0f / (1.0f + expf(-gg))));
                }
                uint16_t* dst = p.C + row * p.ldc + col;
                if (vec && col + n <= p.N) {
                    if (n == 4) *reinterpret_cast<uint2*>(dst) = make_uint2(pack2(h[0], h[1]), pack2(h[2], h[3]));
                    else *reinterpret_cast<uint32_t*>(dst) = pack2(h[0], h[1]);
                } else {
#pragma unroll
                    for (int r = 0; r < n; r++)
                        if (col + r < p.N) dst[r] = f2bf(h[r]);
                }
            }
        }
    } else if constexpr (EPI == kEpiQkv) {
        qkv_tail<FH, FJ, EARLY>(p, tail, row0, nt * BN + wn * TN + 4 * g, res, ops);
    } else {
#pragma unroll
        for (int j = 0; j < FJ; j++) {
            const int64_t col = nt * BN + wn * TN + j * 16 + 4 * g;
            float bias[4] = {0.f, 0.f, 0.f, 0.f};
            if constexpr (EPI == QIE_EPI_STORE) quad_bias(p, col, bias);
#pragma unroll
            for (int i = 0; i < FH; i++) {
                const int64_t row = row0 + i * 16;
                if (row >= p.M) continue;
                const f32x4 v = res[i][j];
                if constexpr (EPI == QIE_EPI_F32) {
                    store_quad_f32(reinterpret_cast<float*>(p.C) + row * p.ldc + col, v, vec, p.N - col);
                } else if constexpr (EPI == QIE_EPI_RESIDUAL) {
                    uint16_t* dst = p.C + row * p.ldc + col;
                    add_quad(dst, quad_before(dst, vec, p.N - col), v, vec, p.N - col);
                } else {
                    const float o[4] = {v[0] + bias[0], v[1] + bias[1], v[2] + bias[2], v[3] + bias[3]};
                    store_quad(p.C + row * p.ldc + col, o, vec, p.N - col);
                }
            }
        }
    }
}

// ---------------------------------------------------------------- the plan
namespace {
template <int EPI, int BM, int BN, int SLOTS>
int launch_mid_t(const GemmParams& p, const mid::Plan& pl, const G8Split& sk, const TailOf<EPI>& tail, hipStream_t st) {
    const void* fn = (const void*)gemm_mid_kernel<EPI, BM, BN, SLOTS>;
    constexpr size_t shm = (size_t)SLOTS * (BM + BN) * 128;
    static bool raised = false;
    if (!raised) {
        QIE_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm));
        raised = true;
    }
    const int tiles = pl.n_mt * pl.n_nt, whole = sk.splitk > 1 ? pl.whole : tiles;
    hipLaunchKernelGGL((gemm_mid_kernel<EPI, BM, BN, SLOTS>), dim3((unsigned)(whole + (tiles - whole) * sk.splitk)), dim3(512), shm,
                       st, p, pl.n_mt, pl.n_nt, band_height(pl.n_mt, BM, BN, 32 * mid::shape(pl.tile).per_cu), whole, sk, tail);
    QIE_LAUNCH_CHECK();
    return 0;
}

template <int EPI>
int launch_mid(const GemmParams& p, const mid::Plan& pl, const G8Split& sk, hipStream_t st, const TailOf<EPI>& tail = {}) {
    switch (pl.tile) {
        case 0: return launch_mid_t<EPI, 64, 64, 5>(p, pl, sk, tail, st);
        case 1: return launch_mid_t<EPI, 64, 128, 3>(p, pl, sk, tail, st);
        case 2: return launch_mid_t<EPI, 128, 64, 3>(p, pl, sk, tail, st);
        case 3: return launch_mid_t<EPI, 128, 128, 4>(p, pl, sk, tail, st);
        case 4: return launch_mid_t<EPI, 192, 128, 4>(p, pl, sk, tail, st);
        case 5: return launch_mid_t<EPI, 256, 128, 3>(p, pl, sk, tail, st);
        case 6: return launch_mid_t<EPI, 320, 64, 3>(p, pl, sk, tail, st);
        case 7: return launch_mid_t<EPI, 320, 128, 2>(p, pl, sk, tail, st);
        case 8: return launch_mid_t<EPI, 128, 160, 4>(p, pl, sk, tail, st);
        case 9: return launch_mid_t<EPI, 192, 160, 3>(p, pl, sk, tail, st);
        case 10: return launch_mid_t<EPI, 256, 160, 3>(p, pl, sk, tail, st);
        default: return launch_mid_t<EPI, 320, 160, 2>(p, pl, sk, tail, st);
    }
}
}  // namespace

int gemm_mid(const qie_linear_args* a, const GemmParams& p, const QkvTail* tail, hipStream_t st, bool* launched) {
    *launched = false;
    const mid::Plan pl = mid::choose(a->M, a->epilogue == QIE_EPI_SWIGLU ? 2 * a->N : a->N, a->K, device_cu_count());
    if (pl.tile < 0) return 0;
    G8Split sk{1, nullptr, nullptr};
    const int64_t cut = (int64_t)pl.n_mt * pl.n_nt - pl.whole;
    if (pl.splitk > 1 && cut > 0) {
        const int64_t floats = cut * pl.splitk * mid::shape(pl.tile).bm * mid::shape(pl.tile).bn;
        if (g8_workspace(st, (int)cdiv(floats, 65536), (int)cut, &sk) == 0) sk.splitk = pl.splitk;
    }
    *launched = true;
    if (tail) return launch_mid<kEpiQkv>(p, pl, sk, st, *tail);
    switch (a->epilogue) {
        case QIE_EPI_SWIGLU: return launch_mid<QIE_EPI_SWIGLU>(p, pl, sk, st);
        case QIE_EPI_RESIDUAL: return launch_mid<QIE_EPI_RESIDUAL>(p, pl, sk, st);
        case QIE_EPI_F32: return launch_mid<QIE_EPI_F32>(p, pl, sk, st);
        default: return launch_mid<QIE_EPI_STORE>(p, pl, sk, st);
    }
}

}  // namespace qie
