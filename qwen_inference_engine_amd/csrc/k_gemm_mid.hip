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
//   * 8 waves.  The two 32-deep halves of a k-tile are summed apart, either by waves 0 .. 3 and 4 .. 7 (2 x 2 of them over the tile; they meet
//     in LDS behind the loop) or by every wave (4 x 2) in registers of its own, which needs no meeting: 320 x 160 spent 10 of 100 us on it.
//     The sums are the same bits.  LDS gives 230 B a clock, so how often it is read does not decide;
//   * in turns: waves 4 .. 7 run one barrier behind waves 0 .. 3, on every SIMD one wave's products run while the other's fragments are
//     read.  Which form a tile has is what 184 shapes of 12 projections at 24 to 3,000 rows measured, and for 128, 192 and 256 x 128, that change
//     it with the k-tiles of a part, 300 more.  Those three in step with halves by register / in turns with halves by wave, us: 128 rows a tile, 222
//     rows, K = 1,792, 23.6 / 24.5, 232 rows, 3,072, 33.7 / 35.5, 336 rows, 4,096, 45.2 / 44.8, 885 rows, 2,048, 21.7 / 22.3, 846 rows, 3,584, 39.1 / 38.1,
//     303 rows, 8,192, 80.9 / 78.2; 192, 395 rows, 256, 8.7 / 10.6, 272 rows, 896, 17.8 / 19.0, 830 rows, 2,048, 30.4 / 28.7; 256, 217 rows, 512, 15.6 / 18.4, 677 rows, 1,536, 31.1 / 31.3, 667 rows, 3,584,
//     59.5 / 53.9.  One row tile: 104 rows, 2,048, 25.9 / 27.6, 72 rows, 5,120, 54.8 / 56.8, 176 rows, 2,048, 36.2 / 38.2, 138 rows, 5,120, 70.3 / 73.9,
//     145 rows, 8,192, 116.9 / 108.7, in two parts of it 66.0 / 67.3;
//   * 320 rows: W of one k-tile more than A in flight (its lines come from HBM, A's mostly from L2, and a CU returns them in order): the
//     staging alone 80 -> 69 us at 320 x 160;
//   * split-K over workgroups where the tiles do not fill the chip (fp32 slabs, the last arriver sums them in part order: gemm8_kernel's
//     protocol, the result does not depend on arrival order).  A wave's share of a tile meets by itself, with a ticket of its own: the
//     shares' last arrivers are spread over the parts' CUs, and none waits for its workgroup (301 rows, O, 25.4 -> 22.9 us);
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

template <int EPI, int BM, int BN, int SA, int SW, int KW, bool TURNS>
__global__ __launch_bounds__(512) void gemm_mid_kernel(GemmParams p, int n_mt, int n_nt, int gm, int whole, G8Split sk, TailOf<EPI> tail) {
#pragma clang fp contract(off)
    constexpr int HV = 2 / KW;   // halves of a k-tile that a wave has: KW 1, waves as 4 (M) x 2 (N), both; KW 2, 2 x 2 x the halves
    constexpr int TM = BM / (4 / KW), TN = BN / 2, FI = TM / 16, FJ = TN / 16;   // a wave's tile
    constexpr int A_SLOT = BM * 128, W_SLOT = BN * 128, W_BASE = SA * A_SLOT;
    // LDS-DMA instructions (8 rows each) per wave and k-tile; where the waves don't share W's evenly, the first MORE have one more
    constexpr int AIW = BM / 64, WIW = (BN / 8 + 7) / 8, MORE = BN / 8 % 8;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = KW == 2 ? wave >> 2 : 0, wm = KW == 2 ? (wave >> 1) & 1 : wave >> 1, wn = wave & 1;
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

    const int nk_all = (int)(p.K >> 6);
    const int kb = quotient(part * nk_all, parts), nk = quotient((part + 1) * nk_all, parts) - kb;   // this part's k-tiles [kb, kb + nk)

    // instruction i of this wave fills the slot's rows 8 b .. 8 b + 7, b = 8 i + wave: lane -> row 8 b + (lane >> 3),
    // LDS chunk lane & 7, which holds the source's chunk (lane & 7) ^ swz(row)
    uint32_t a_off[AIW];   // bytes behind the tile's first row
    const uint16_t* w_src[WIW];
    const int r0 = 8 * wave + (lane >> 3), cs = ((lane & 7) ^ g8_swz(r0)) * 8;   // (64 rows on: the same chunk)
    const int64_t k0 = (int64_t)kb * mid::BK + cs;
#pragma unroll
    for (int i = 0; i < AIW; i++) {
        int64_t ar = m0 + r0 + 64 * i;
        ar = ar < p.M ? ar : p.M - 1;   // rows past M: re-read row M - 1, never stored
        a_off[i] = (uint32_t)(ar - m0) * (uint32_t)p.lda * 2 + (uint32_t)cs * 2;
    }
#pragma unroll
    for (int i = 0; i < WIW; i++) {
        if (MORE && i == WIW - 1 && wave >= MORE) break;   // uniform
        w_src[i] = mid_wrow<EPI, BN>(p, nt, r0 + 64 * i) + k0;
    }
    constexpr int FR = FI / KW;   // a wave's rows of the result, in fragments
    const int wrow = wm * TM + wk * (FR * 16) + fr;
    // kEpiQkv of small tiles: its operands are on their way before the first k-tile
    const int64_t row0 = m0 + wrow;
    constexpr bool EARLY = EPI == kEpiQkv && FR * FJ <= 8;
    [[maybe_unused]] QkvOps<FR> ops[EARLY ? FJ : 1];
    if constexpr (EARLY) {
#pragma unroll
        for (int j = 0; j < FJ; j++) qkv_load(p, tail, row0, nt * BN + wn * TN + 16 * j + 4 * g, ops[j]);
        __builtin_amdgcn_sched_barrier(0);
    }
    const uint16_t* a_at = p.A + m0 * p.lda + (int64_t)kb * mid::BK;
    auto stage_a = [&](int kt, int slot) {
#pragma unroll
        for (int i = 0; i < AIW; i++) glds16(reinterpret_cast<const unsigned char*>(a_at + (int64_t)kt * mid::BK) + a_off[i], smem + slot * A_SLOT + wave * 1024 + i * 8192);
    };
    auto stage_w = [&](int kt, int slot) {
#pragma unroll
        for (int i = 0; i < WIW; i++) {
            if (MORE && i == WIW - 1 && wave >= MORE) break;
            glds16(w_src[i] + (int64_t)kt * mid::BK, smem + W_BASE + slot * W_SLOT + wave * 1024 + i * 8192);
        }
    };

    // sums of either half of every k-tile
    f32x4 acc[HV][FI][FJ];
#pragma unroll
    for (int s = 0; s < HV; s++)
#pragma unroll
        for (int i = 0; i < FI; i++)
#pragma unroll
            for (int j = 0; j < FJ; j++) acc[s][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // step t stages A of k-tile t + SA - 1, then W of t + SW - 1: the steps before the first
#pragma unroll
    for (int t = 1 - SW; t < 0; t++) {
        if (t + SA - 1 >= 0 && t + SA - 1 < nk) stage_a(t + SA - 1, t + SA - 1);
        if (t + SW - 1 < nk) stage_w(t + SW - 1, t + SW - 1);
    }
    constexpr int YOUNG = SA - 2, AHEAD_W = SW > SA ? 1 : 0;   // k-tiles, and W's of one more, that fly behind the one waited for
    static_assert(SW >= SA, "A of a k-tile is staged no earlier than its W");
    auto landed = [&](bool steady) {   // the k-tile after which `steady` steps were staged
        if (steady && (MORE == 0 || wave < MORE)) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((AIW + WIW) * YOUNG + WIW * AHEAD_W) : "memory");
        else if (steady) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((AIW + WIW - 1) * YOUNG + (WIW - 1) * AHEAD_W) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };
    auto bar = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    auto frag = [&](const unsigned char* buf, int row, int s) {
        return *reinterpret_cast<const bf16x8*>(buf + row * 128 + (((4 * s + g) ^ g8_swz(row)) * 16));
    };
    int sa = 0, sw = 0, fill_a = SA - 1, fill_w = SW - 1;
    auto advance = [&]() {
        sa = sa + 1 == SA ? 0 : sa + 1;
        fill_a = fill_a + 1 == SA ? 0 : fill_a + 1;
        sw = sw + 1 == SW ? 0 : sw + 1;
        fill_w = fill_w + 1 == SW ? 0 : fill_w + 1;
    };
    if constexpr (TURNS) {
        // Waves 4 .. 7 run one barrier behind waves 0 .. 3: on every SIMD one wave reads its fragments while the other's products run.
        // A slot's reads end before the barrier behind them, so it is staged anew from the next step on.
        constexpr int PH = FI * FJ * HV <= 32 ? 1 : HV, HS = HV / PH;   // phases a k-tile: both halves' fragments at once where registers hold them
        const bool late = wave >= 4;
        landed(SW - 1 <= nk);
        bar();
        if (late) bar();
        for (int t = 0; t < nk; t++) {
            const unsigned char *a_buf = smem + sa * A_SLOT, *w_buf = smem + W_BASE + sw * W_SLOT;
#pragma unroll
            for (int ph = 0; ph < PH; ph++) {
                bf16x8 fa[HS][FI], fb[HS][FJ];
#pragma unroll
                for (int h = 0; h < HS; h++) {
#pragma unroll
                    for (int j = 0; j < FJ; j++) fb[h][j] = frag(w_buf, wn * TN + j * 16 + fr, wk + ph * HS + h);
#pragma unroll
                    for (int i = 0; i < FI; i++) fa[h][i] = frag(a_buf, wm * TM + i * 16 + fr, wk + ph * HS + h);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (ph == 0) {
                    if (t + SA - 1 < nk) stage_a(t + SA - 1, fill_a);
                    if (t + SW - 1 < nk) stage_w(t + SW - 1, fill_w);
                }
                if (ph == PH - 1 && late && t + 1 < nk) landed(t + SW <= nk);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                bar();
                __builtin_amdgcn_s_setprio(1);
#pragma unroll
                for (int h = 0; h < HS; h++)
#pragma unroll
                    for (int i = 0; i < FI; i++)
#pragma unroll
                        for (int j = 0; j < FJ; j++)
                            acc[ph * HS + h][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[h][j], fa[h][i], acc[ph * HS + h][i][j], 0, 0, 0);   // W Aᵀ
                __builtin_amdgcn_s_setprio(0);
                __builtin_amdgcn_sched_barrier(0);
                if (ph == PH - 1 && !late && t + 1 < nk) landed(t + SW <= nk);
                bar();
            }
            advance();
        }
        if (!late) bar();
    } else {
        for (int t = 0; t < nk; t++) {
            // k-tile t has landed (what was staged behind it may still fly), and every wave is done with the slots of t - 1
            landed(t + SW - 1 <= nk);
            bar();
            if (t + SA - 1 < nk) stage_a(t + SA - 1, fill_a);
            if (t + SW - 1 < nk) stage_w(t + SW - 1, fill_w);
            const unsigned char *a_buf = smem + sa * A_SLOT, *w_buf = smem + W_BASE + sw * W_SLOT;
            constexpr int HS = FI * FJ <= 10 ? HV : 1;      // halves whose fragments are read together
            constexpr int AHEAD = FI * FJ > 20 ? 2 : FI;    // few registers left: two A fragments on their way while one is multiplied
#pragma unroll
            for (int s0 = 0; s0 < HV; s0 += HS) {
                bf16x8 fa[HS][FI], fb[HS][FJ];
#pragma unroll
                for (int h = 0; h < HS; h++) {
#pragma unroll
                    for (int j = 0; j < FJ; j++) fb[h][j] = frag(w_buf, wn * TN + j * 16 + fr, wk + s0 + h);
#pragma unroll
                    for (int i = 0; i < AHEAD; i++) fa[h][i] = frag(a_buf, wm * TM + i * 16 + fr, wk + s0 + h);
                }
                if (HS == 2) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int h = 0; h < HS; h++)
#pragma unroll
                    for (int i = 0; i < FI; i++) {
                        if (i + AHEAD < FI) fa[h][i + AHEAD] = frag(a_buf, wm * TM + (i + AHEAD) * 16 + fr, wk + s0 + h);
                        if (AHEAD < FI) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int j = 0; j < FJ; j++)
                            acc[s0 + h][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[h][j], fa[h][i], acc[s0 + h][i][j], 0, 0, 0);   // W Aᵀ
                        if (AHEAD < FI) __builtin_amdgcn_sched_barrier(0);
                    }
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // this wave's reads of the slots are done
            __builtin_amdgcn_sched_barrier(0);
            advance();
        }
    }
    f32x4 res[FR][FJ];
    if constexpr (KW == 1) {
#pragma unroll
        for (int i = 0; i < FR; i++)
#pragma unroll
            for (int j = 0; j < FJ; j++) res[i][j] = acc[0][i][j] + acc[1][i][j];
    } else {   // waves w and w ^ 4 hold the same tile; each keeps half of its rows
        f32x4* ex = reinterpret_cast<f32x4*>(smem);
        static_assert(8 * FR * FJ * 1024 <= (SA * BM + SW * BN) * 128, "exchange area");
        __syncthreads();
#pragma unroll
        for (int i = 0; i < FR; i++)
#pragma unroll
            for (int j = 0; j < FJ; j++) {
                ex[((wave * FR + i) * FJ + j) * 64 + lane] = wk == 0 ? acc[0][FR + i][j] : acc[0][i][j];
                res[i][j] = wk == 0 ? acc[0][i][j] : acc[0][FR + i][j];
            }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < FR; i++)
#pragma unroll
            for (int j = 0; j < FJ; j++) res[i][j] = res[i][j] + ex[(((wave ^ 4) * FR + i) * FJ + j) * 64 + lane];
    }

    if constexpr (EPI == kEpiParts) {   // rows past M lie behind the part's end, columns past N are moved there
        const int ldp = (int)p.N * 4;
        const auto rs = __builtin_amdgcn_make_buffer_rsrc(sk.slab + (int64_t)part * p.M * p.N, (short)0, (int)p.M * ldp, 0x00020000);
#pragma unroll
        for (int j = 0; j < FJ; j++) {
            const int col = (int)nt * BN + wn * TN + 16 * j + 4 * g;
#pragma unroll
            for (int i = 0; i < FR; i++)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_g8, res[i][j]), rs, col < p.N ? ((int)m0 + wrow + 16 * i) * ldp + col * 4 : 1 << 31, 0, 0);
        }
        return;
    }

    // The tile's part of C as a buffer: rows past M lie behind its end, and so do columns past N, moved there by `at`; loads from there give 0,
    // stores do nothing.
    constexpr int OUT_BN = EPI == QIE_EPI_SWIGLU ? BN / 2 : BN, SZ = EPI == QIE_EPI_F32 ? 4 : 2, OUTSIDE = 1 << 31;
    const bool quads = p.vec != 0 && (p.N & 3) == 0;   // uniform
    const int ld = (int)p.ldc * SZ, left = (int)(p.N - nt * OUT_BN < OUT_BN ? p.N - nt * OUT_BN : OUT_BN);   // bytes of a row; columns
    const auto c_rs = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<unsigned char*>(p.C) + (m0 * p.ldc + nt * OUT_BN) * SZ, (short)0,
                                                        ((int)(p.M - m0 < BM ? p.M - m0 : BM) - 1) * ld + left * SZ, 0x00020000);
    const int c_row = wrow * ld;
    auto at = [&](int i, int col) { return (col < left ? c_row + col * SZ : OUTSIDE) + i * 16 * ld; };
    auto put = [&](int i, int col, int n, const float (&v)[4]) {   // columns col .. col + n - 1 of the tile
        if (quads) {
            if (n == 4) __builtin_amdgcn_raw_buffer_store_b64(u32x2_g8{pack2(v[0], v[1]), pack2(v[2], v[3])}, c_rs, at(i, col), 0, 0);
            else __builtin_amdgcn_raw_buffer_store_b32(pack2(v[0], v[1]), c_rs, at(i, col), 0, 0);
        } else {
#pragma unroll
            for (int r = 0; r < n; r++) __builtin_amdgcn_raw_buffer_store_b16(f2bf(v[r]), c_rs, at(i, col + r), 0, 0);
        }
    };
    const int col0 = wn * TN + 4 * g;
    // residuals: all on their way at once; ahead of the parts' sum where registers hold both
    [[maybe_unused]] uint2 before[FR][FJ];
    [[maybe_unused]] auto load_before = [&]() {
        if (quads) {
#pragma unroll
            for (int i = 0; i < FR; i++)
#pragma unroll
                for (int j = 0; j < FJ; j++)
                    before[i][j] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(c_rs, at(i, col0 + 16 * j), 0, 0));
        } else {
#pragma unroll
            for (int i = 0; i < FR; i++)
#pragma unroll
                for (int j = 0; j < FJ; j++) {
                    uint32_t h[4];
#pragma unroll
                    for (int r = 0; r < 4; r++) h[r] = __builtin_amdgcn_raw_buffer_load_b16(c_rs, at(i, col0 + 16 * j + r), 0, 0);
                    before[i][j] = make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
                }
        }
    };
    constexpr bool BOTH = FR * FJ <= 16;
    if constexpr (EPI == QIE_EPI_RESIDUAL && BOTH) load_before();

    constexpr bool SPLITS = BN != 160;   // (mid::WIDE: whole, or in parts that another launch adds up)
    if (SPLITS && parts > 1) {   // uniform.  A wave's share of the tile meets by itself: no wave waits for the others of its workgroup
        constexpr int SLAB = BM * BN;   // floats
        const int64_t tb = (int64_t)ct * parts;
        const int slab_at = (wave * FR * FJ * 64 + lane) * 16;
        const auto rs = __builtin_amdgcn_make_buffer_rsrc(sk.slab + (tb + part) * SLAB, (short)0, SLAB * 4, 0x00020000);
#pragma unroll
        for (int i = 0; i < FR; i++)
#pragma unroll
            for (int j = 0; j < FJ; j++)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_g8, res[i][j]), rs, slab_at + (i * FJ + j) * 1024, 0, 16);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // stored
        unsigned* cnt = sk.cnt + (ct * 8 + wave) * G8_TICKET;
        unsigned old = 0;
        if (lane == 0) old = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        old = __builtin_amdgcn_readfirstlane(old);
        if (old != (unsigned)parts - 1) return;   // uniform
        asm volatile("" ::: "memory");
        // part order, this part's own from its registers: independent of who arrived last; as many of the others' on their way as registers
        // hold (small tiles: of two workgroups a CU)
        constexpr int FLY = KW == 2 ? 16 : FR * FJ <= 16 ? 24 : 12, IG = FR * FJ <= 8 ? FR : 1, QN = FLY / (IG * FJ) < 6 ? FLY / (IG * FJ) : 6;   // fragments; rows of them; parts
#pragma unroll
        for (int i0 = 0; i0 < FR; i0 += IG) {
            f32x4 sum[IG][FJ];
            for (int q0 = 0; q0 < parts; q0 += QN) {
                f32x4 v[QN][IG][FJ];
#pragma unroll
                for (int u = 0; u < QN; u++) {
                    if (q0 + u >= parts || q0 + u == part) continue;
                    const auto rq = __builtin_amdgcn_make_buffer_rsrc(sk.slab + (tb + q0 + u) * SLAB, (short)0, SLAB * 4, 0x00020000);
#pragma unroll
                    for (int i = 0; i < IG; i++)
#pragma unroll
                        for (int j = 0; j < FJ; j++)
                            v[u][i][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rq, slab_at + ((i0 + i) * FJ + j) * 1024, 0, 16));
                }
#pragma unroll
                for (int u = 0; u < QN; u++) {
                    if (q0 + u >= parts) break;
#pragma unroll
                    for (int i = 0; i < IG; i++)
#pragma unroll
                        for (int j = 0; j < FJ; j++) {
                            const f32x4 w = q0 + u == part ? res[i0 + i][j] : v[u][i][j];
                            sum[i][j] = q0 + u == 0 ? w : sum[i][j] + w;
                        }
                }
            }
#pragma unroll
            for (int i = 0; i < IG; i++)
#pragma unroll
                for (int j = 0; j < FJ; j++) res[i0 + i][j] = sum[i][j];
        }
        if (lane == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // ---------------- epilogue.  D = W Aᵀ: a lane holds row m = lane & 15 and the columns 4 g .. 4 g + 3 of a fragment, one
    // 8- (fp32: 16-) byte store where C's rows allow it
    if constexpr (EPI == QIE_EPI_RESIDUAL && !BOTH) load_before();
    if constexpr (EPI == QIE_EPI_SWIGLU) {
#pragma unroll
        for (int m = 0; m < (FJ + 1) / 2; m++) {
            constexpr int PAIRS = FJ / 2;
            const int n = m < PAIRS ? 4 : 2;   // outputs
#pragma unroll
            for (int i = 0; i < FR; i++) {
                float h[4];
#pragma unroll
                for (int r = 0; r < n; r++) {
                    const f32x4 v = res[i][2 * m + r / 2];
                    const float gg = rbf(v[r & 1]);
                    const float uu = rbf(v[2 + (r & 1)]);
                    h[r] = uu * rbf(gg * (1.0f / (1.0f + expf(-gg))));
                }
                put(i, (TN / 2) * wn + 16 * m + n * g, n, h);
            }
        }
    } else if constexpr (EPI == kEpiQkv) {
        qkv_tail<FR, FJ, EARLY>(p, tail, row0, nt * BN + wn * TN + 4 * g, res, ops);
    } else {
#pragma unroll
        for (int j = 0; j < FJ; j++) {
            float bias[4] = {0.f, 0.f, 0.f, 0.f};
            if constexpr (EPI == QIE_EPI_STORE) quad_bias(p, nt * BN + col0 + 16 * j, bias);
#pragma unroll
            for (int i = 0; i < FR; i++) {
                const f32x4 v = res[i][j];
                if constexpr (EPI == QIE_EPI_F32) {
                    if (quads) {
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_g8, v), c_rs, at(i, col0 + 16 * j), 0, 0);
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; r++) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[r]), c_rs, at(i, col0 + 16 * j + r), 0, 0);
                    }
                } else {
                    float o[4] = {v[0] + bias[0], v[1] + bias[1], v[2] + bias[2], v[3] + bias[3]};
                    if constexpr (EPI == QIE_EPI_RESIDUAL) sum_quad(before[i][j], v, o);
                    put(i, col0 + 16 * j, 4, o);
                }
            }
        }
    }
}

// ---------------------------------------------------------------- the plan
namespace {
template <int EPI, int BM, int BN, int SA, int SW, int KW, bool TURNS>
int launch_mid_t(const GemmParams& p, const mid::Plan& pl, const G8Split& sk, const TailOf<EPI>& tail, hipStream_t st) {
    const void* fn = (const void*)gemm_mid_kernel<EPI, BM, BN, SA, SW, KW, TURNS>;
    constexpr size_t shm = (size_t)(SA * BM + SW * BN) * 128;
    static bool raised = false;
    if (!raised) {
        QIE_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm));
        raised = true;
    }
    const int tiles = pl.n_mt * pl.n_nt, whole = EPI == kEpiParts ? 0 : sk.splitk > 1 ? pl.whole : tiles;
    hipLaunchKernelGGL((gemm_mid_kernel<EPI, BM, BN, SA, SW, KW, TURNS>), dim3((unsigned)(whole + (tiles - whole) * sk.splitk)), dim3(512), shm,
                       st, p, pl.n_mt, pl.n_nt, band_height(pl.n_mt, BM, BN, 32 * mid::shape(pl.tile).per_cu), whole, sk, tail);
    QIE_LAUNCH_CHECK();
    return 0;
}

template <int EPI>
int launch_mid(const GemmParams& p, const mid::Plan& pl, const G8Split& sk, hipStream_t st, const TailOf<EPI>& tail = {}) {
    // one row tile, and a part of K that is not too long: what its workgroups wait for is their weights from memory, which the form in turns is no help to
    const bool streams = pl.n_mt == 1 && p.K < 6144 * pl.splitk;
    switch (pl.tile) {
        case 0: return launch_mid_t<EPI, 64, 64, 5, 5, 2, false>(p, pl, sk, tail, st);
        case 1: return launch_mid_t<EPI, 64, 128, 3, 3, 2, false>(p, pl, sk, tail, st);
        case 2: return launch_mid_t<EPI, 128, 64, 3, 3, 2, false>(p, pl, sk, tail, st);
        case 3:
            if (p.K < (pl.n_mt <= 4 ? 4096 : 2304) * pl.splitk || streams) return launch_mid_t<EPI, 128, 128, 4, 4, 1, false>(p, pl, sk, tail, st);
            return launch_mid_t<EPI, 128, 128, 4, 4, 2, true>(p, pl, sk, tail, st);
        case 4:
            if (p.K < 1280 || streams) return launch_mid_t<EPI, 192, 128, 4, 4, 1, false>(p, pl, sk, tail, st);
            return launch_mid_t<EPI, 192, 128, 4, 4, 2, true>(p, pl, sk, tail, st);
        case 5:
            if (p.K < 1792 || streams) return launch_mid_t<EPI, 256, 128, 3, 3, 1, false>(p, pl, sk, tail, st);
            return launch_mid_t<EPI, 256, 128, 3, 3, 2, true>(p, pl, sk, tail, st);
        case 6: return launch_mid_t<EPI, 320, 64, 3, 3, 1, false>(p, pl, sk, tail, st);
        case 7: return launch_mid_t<EPI, 320, 128, 2, 4, 1, true>(p, pl, sk, tail, st);
        case 8: return launch_mid_t<EPI, 128, 160, 4, 4, 1, true>(p, pl, sk, tail, st);
        case 9: return launch_mid_t<EPI, 192, 160, 3, 3, 1, true>(p, pl, sk, tail, st);
        case 10: return launch_mid_t<EPI, 256, 160, 3, 3, 1, true>(p, pl, sk, tail, st);
        default: return launch_mid_t<EPI, 320, 160, 2, 3, 1, false>(p, pl, sk, tail, st);
    }
}
}  // namespace

static int run_mid(int epi, const GemmParams& p, const mid::Plan& pl, const QkvTail* tail, hipStream_t st) {
    G8Split sk{1, nullptr, nullptr};
    const int64_t cut = (int64_t)pl.n_mt * pl.n_nt - pl.whole;
    if (pl.splitk > 1 && cut > 0) {
        const int64_t floats = cut * pl.splitk * mid::shape(pl.tile).bm * mid::shape(pl.tile).bn;
        if (g8_workspace(st, (int)cdiv(floats, 65536), (int)cut * 8 * G8_TICKET, &sk) == 0) sk.splitk = pl.splitk;
    }
    if (tail) return launch_mid<kEpiQkv>(p, pl, sk, st, *tail);
    switch (epi) {
        case QIE_EPI_SWIGLU: return launch_mid<QIE_EPI_SWIGLU>(p, pl, sk, st);
        case QIE_EPI_RESIDUAL: return launch_mid<QIE_EPI_RESIDUAL>(p, pl, sk, st);
        case QIE_EPI_F32: return launch_mid<QIE_EPI_F32>(p, pl, sk, st);
        default: return launch_mid<QIE_EPI_STORE>(p, pl, sk, st);
    }
}

int gemm_mid(const qie_linear_args* a, const GemmParams& p, const QkvTail* tail, hipStream_t st, bool* launched) {
    *launched = false;
    const mid::Plan pl = mid::choose(a->M, a->epilogue == QIE_EPI_SWIGLU ? 2 * a->N : a->N, a->K, device_cu_count());
    if (pl.tile < 0 || !mid::strides_fit(a->ldx, a->ldy)) return 0;
    *launched = true;
    return run_mid(a->epilogue, p, pl, tail, st);
}

int gemm_mid_parts(const GemmParams& p, int tile, const G8Split& sk, hipStream_t st) {
    mid::Plan pl{tile, 0, sk.splitk, (int)cdiv(p.M, mid::shape(tile).bm), (int)cdiv(p.N, mid::shape(tile).bn), 0.f};
    return launch_mid<kEpiParts>(p, pl, sk, st);
}

int gemm_mid_rest(int epi, const GemmParams& p, hipStream_t st) {
    return run_mid(epi, p, mid::best(p.M, epi == QIE_EPI_SWIGLU ? 2 * p.N : p.N, p.K, device_cu_count()), nullptr, st);
}

}  // namespace qie
