// k_gemm_few.hip — MFMA bf16 GEMM for prompts whose tiles leave the chip's CUs mostly waiting: a wave has a share of K to itself.
//
//   C[M, N] = A[M, K] . W[N, K]^T, fp32 accumulation, the epilogues of k_gemm.hip, or the sums of parts of K
//
// k_gemm_mid.hip's workgroup walks K together, one barrier per 64 of it: 0.29 us a k-tile for 64 x 64 outputs however little of them there is
// (Qwen2-0.5B's QKV at 24 rows 6.4 us, 6.2 with its weights already in L2; the launch alone 2.0).  What bounds such a launch is the bytes that one CU
// stages and the steps ahead of its first product, so here:
//   * tiles of 32 x 16 to 64 x 64: more CUs, fewer bytes for each;
//   * a workgroup of 4 waves, each with the 64-deep chunks wave, wave + 4, ... of the tile's K, which it stages itself by LDS-DMA (whole 128-byte
//     lines, 8 rows an instruction) into a ring of its own and multiplies without a look at the others': no barrier before the tiles meet in
//     LDS at the end, where a wave sums a fragment (SwiGLU: a gate and an up fragment) of all and runs its epilogue;
//   * W A^T as in k_gemm.hip: a lane ends with four neighbouring columns of a row.
// us, k_gemm_mid.hip / this: Qwen2-0.5B QKV 24 rows 6.4 / 4.3, 113 rows 6.8 / 4.5, 256 rows 6.8 / 5.6; 1,536 -> 2,048 at 113 rows 8.1 / 5.4; Qwen3-14B QKV
// at 24 rows 19.0 / 16.0; Qwen2-7B gate / up at 24 rows 53.4 / 48.8 (and no longer behind from 33 rows on: it reads x for every 16 or 32 of W's rows).
// Fragments straight from memory into registers instead of LDS, 64 bytes of a row an instruction, ran at half the rate.
// Sums: chains of a wave's share of K, the shares in wave order.
#include "gemm_impl.hpp"
#include "gemm_plan.hpp"

#include <algorithm>

namespace qie {


// FI, FJ: fragments of 16 rows of A, of 16 weight rows (SwiGLU: gate and up in turn); SLOTS of a wave's ring; NT: weights that one row tile reads
template <int EPI, int FI, int FJ, int SLOTS, bool NT>
__global__ __launch_bounds__(64 * few::WAVES) void gemm_few_kernel(GemmParams p, int n_mt, int n_nt, int parts, float* slab, TailOf<EPI> tail) {
#pragma clang fp contract(off)
    constexpr int NW = few::WAVES, BM = 16 * FI, BN = 16 * FJ;
    constexpr bool GATED = EPI == QIE_EPI_SWIGLU;
    constexpr int SLOT = (BM + BN) * 128, IPC = (BM + BN) / 8;   // bytes and LDS-DMA instructions of a chunk
    static_assert(!GATED || FJ % 2 == 0, "gate and up fragments in pairs");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, g = lane >> 4;
    // neighbours (the row tiles of a weight tile) on one XCD, parts slowest
    const int nwg = gridDim.x, orig = blockIdx.x, q8 = nwg >> 3, r8 = nwg & 7, xcd = orig & 7;
    const int wid = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + (orig >> 3);
    const int tiles = n_mt * n_nt, part = quotient(wid, tiles), tile = wid - part * tiles, nt = quotient(tile, n_mt), mt = tile - nt * n_mt;
    const int64_t m0 = (int64_t)mt * BM, c0 = (int64_t)nt * (GATED ? BN / 2 : BN);
    const int chunks = (int)(p.K >> 6), kb = quotient(part * chunks, parts), n = quotient((part + 1) * chunks, parts) - kb;
    const int mine = n > wave ? (n - wave + NW - 1) / NW : 0;   // chunks kb + wave + NW i of this wave

    // A's and the weights' rows of the tile as buffers (few::bytes_of).  A tile lies in one weight segment (few::choose).
    const int rows = (int)(p.M - m0 < BM ? p.M - m0 : BM);
    const uint16_t* a0 = p.A + m0 * p.lda;
    const int64_t seg = GATED || c0 < p.n0 ? 0 : c0 < p.n01 ? p.n0 : p.n01, end = GATED ? p.N : c0 < p.n0 ? p.n0 : c0 < p.n01 ? p.n01 : p.N;
    const uint16_t* w0 = (GATED || c0 < p.n0 ? p.w0 : c0 < p.n01 ? p.w1 : p.w2) + (c0 - seg) * p.K;
    const uint16_t* w1 = GATED ? p.w1 + c0 * p.K : w0;
    const int left = (int)(end - c0 < (GATED ? BN / 2 : BN) ? end - c0 : (GATED ? BN / 2 : BN));
    auto rsrc = [](const void* base, uint32_t bytes) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000); };

    // The fragments that this wave will sum, and what kEpiQkv loads for them ahead of the first chunk
    constexpr int PJ = GATED ? 2 : 1, UNITS = FI * FJ / PJ, ROUNDS = (UNITS + NW - 1) / NW;
    auto unit_row = [&](int u) { return m0 + 16 * (u / (FJ / PJ)) + fr; };
    auto unit_col = [&](int u) { return c0 + 16 * (u % (FJ / PJ)) + 4 * g; };
    constexpr bool EARLY = EPI == kEpiQkv && ROUNDS <= 2;
    [[maybe_unused]] QkvOps<1> ops[EARLY ? ROUNDS : 1][1];
    if constexpr (EARLY) {
#pragma unroll
        for (int r = 0; r < ROUNDS; r++) qkv_load(p, tail, unit_row(r * NW + wave), unit_col(r * NW + wave), ops[r][0]);
        __builtin_amdgcn_sched_barrier(0);
    }

    // instruction b fills the slot's rows 8 b ..: lane -> row 8 b + (lane >> 3), LDS piece lane & 7, which holds the source's piece
    // (lane & 7) ^ swz(row); the swizzle of rows 8 on differs in one bit
    unsigned char* ring = smem + wave * (SLOTS * SLOT);
    const int dr = lane >> 3, piece[2] = {((lane & 7) ^ g8_swz(dr)) * 16, ((lane & 7) ^ g8_swz(dr + 8)) * 16};
    const uint32_t a_bytes = few::bytes_of(rows, p.lda, p.K), w_bytes = few::bytes_of(left, p.K, p.K);
    uint32_t a_at[BM / 8], w_at[BN / 8];
#pragma unroll
    for (int b = 0; b < BM / 8; b++) a_at[b] = few::row_at(8 * b + dr, p.lda) + piece[b & 1];
#pragma unroll
    for (int b = 0; b < BN / 8; b++) w_at[b] = few::row_at(8 * (GATED ? b / 4 * 2 + (b & 1) : b) + dr, p.K) + piece[b & 1];
    auto load = [&](int slot, int i) {
        const bool on = i < mine;   // uniform; off: buffers of no bytes, so that every wait is a counted one
        const int k = (kb + wave + NW * i) * 128;
        const auto ra = rsrc(a0, on ? a_bytes : 0u), r0 = rsrc(w0, on ? w_bytes : 0u), r1 = GATED ? rsrc(w1, on ? w_bytes : 0u) : r0;
        unsigned char* dst = ring + slot * SLOT;
#pragma unroll
        for (int b = 0; b < BN / 8; b++) buffer_lds16<NT>(GATED && (b & 2) ? r1 : r0, dst + b * 1024, w_at[b], k);
#pragma unroll
        for (int b = 0; b < BM / 8; b++) buffer_lds16<false>(ra, dst + BN * 128 + b * 1024, a_at[b], k);
    };
    f32x4 acc[FI][FJ];
#pragma unroll
    for (int i = 0; i < FI; i++)
#pragma unroll
        for (int j = 0; j < FJ; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < SLOTS; s++) load(s, s);
    __builtin_amdgcn_sched_barrier(0);
    auto frag = [&](const unsigned char* buf, int row, int s) { return *reinterpret_cast<const bf16x8*>(buf + row * 128 + (((4 * s + g) ^ g8_swz(row)) * 16)); };
    int slot = 0;
    for (int i = 0; i < mine; i++) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((SLOTS - 1) * IPC) : "memory");   // chunk i has landed
        __builtin_amdgcn_sched_barrier(0);
        const unsigned char *w_buf = ring + slot * SLOT, *a_buf = w_buf + BN * 128;
        bf16x8 fa[2][FI], fb[2][FJ];
#pragma unroll
        for (int s = 0; s < 2; s++) {
#pragma unroll
            for (int j = 0; j < FJ; j++) fb[s][j] = frag(w_buf, 16 * j + fr, s);
#pragma unroll
            for (int a = 0; a < FI; a++) fa[s][a] = frag(a_buf, 16 * a + fr, s);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // read: the slot is free
        __builtin_amdgcn_sched_barrier(0);
        load(slot, i + SLOTS);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int a = 0; a < FI; a++)
#pragma unroll
                for (int j = 0; j < FJ; j++) acc[a][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[s][j], fa[s][a], acc[a][j], 0, 0, 0);   // W Aᵀ
        slot = slot + 1 == SLOTS ? 0 : slot + 1;
    }
    // the waves' shares meet where the rings were: the last loads (of nothing) are done, and every wave's reads
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    f32x4(*red)[FI * FJ][64] = reinterpret_cast<f32x4(*)[FI * FJ][64]>(smem);
#pragma unroll
    for (int i = 0; i < FI; i++)
#pragma unroll
        for (int j = 0; j < FJ; j++) red[wave][i * FJ + j][lane] = acc[i][j];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) {
        const int u = r * NW + wave;   // uniform
        if (UNITS % NW != 0 && u >= UNITS) break;
        f32x4 v[PJ];
#pragma unroll
        for (int h = 0; h < PJ; h++) {
            v[h] = red[0][u * PJ + h][lane];
#pragma unroll
            for (int w = 1; w < NW; w++) v[h] = v[h] + red[w][u * PJ + h][lane];
        }
        const int64_t row = unit_row(u), col = unit_col(u);
        if constexpr (EPI == kEpiQkv) {
            const f32x4 one[1][1] = {{v[0]}};
            qkv_tail<1, 1, EARLY>(p, tail, row, col, one, ops[EARLY ? r : 0]);
        } else {
            if (row >= p.M || col >= p.N) continue;
            const int64_t to_go = p.N - col;
            uint16_t* dst = p.C + row * p.ldc + col;
            if constexpr (EPI == kEpiParts) {
                *reinterpret_cast<f32x4*>(slab + ((int64_t)part * p.M + row) * p.N + col) = v[0];
            } else if constexpr (EPI == QIE_EPI_F32) {
                store_quad_f32(reinterpret_cast<float*>(p.C) + row * p.ldc + col, v[0], p.vec, to_go);
            } else if constexpr (GATED) {
                float h[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float gg = rbf(v[0][e]), uu = rbf(v[PJ - 1][e]);
                    h[e] = uu * rbf(gg * (1.0f / (1.0f + expf(-gg))));
                }
                store_quad(dst, h, p.vec, to_go);
            } else if constexpr (EPI == QIE_EPI_RESIDUAL) {
                add_quad(dst, quad_before(dst, p.vec, to_go), v[0], p.vec, to_go);
            } else {
                float bias[4] = {0.f, 0.f, 0.f, 0.f};
                quad_bias(p, col, bias);
                const float o[4] = {v[0][0] + bias[0], v[0][1] + bias[1], v[0][2] + bias[2], v[0][3] + bias[3]};
                store_quad(dst, o, p.vec, to_go);
            }
        }
    }
}

namespace {
template <int EPI, int FORM, bool NT>
int few_launch(const GemmParams& p, int parts, float* slab, const TailOf<EPI>& tail, hipStream_t st) {
    constexpr few::Form F = few::FORMS[FORM];
    constexpr size_t shm = few::lds(F);
    static_assert(shm <= 160 * 1024, "LDS");
    static bool raised = false;
    if (!raised) {
        QIE_HIP(hipFuncSetAttribute((const void*)gemm_few_kernel<EPI, F.fi, F.fj, F.slots, NT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm));
        raised = true;
    }
    const int n_mt = cdiv(p.M, 16 * F.fi), n_nt = cdiv(p.N, (EPI == QIE_EPI_SWIGLU ? 8 : 16) * F.fj);
    hipLaunchKernelGGL((gemm_few_kernel<EPI, F.fi, F.fj, F.slots, NT>), dim3((unsigned)(n_mt * n_nt * parts)), dim3(64 * few::WAVES), shm, st, p, n_mt, n_nt, parts, slab, tail);
    QIE_LAUNCH_CHECK();
    return 0;
}
// weights with the non-temporal hint where one row tile reads them (Qwen2-7B gate / up at 24 rows 54.6 -> 48.8 us; where two do they come from memory twice)
template <int EPI, int FORM>
int few_one(const GemmParams& p, int parts, float* slab, const TailOf<EPI>& tail, hipStream_t st) {
    return p.M <= 16 * few::FORMS[FORM].fi ? few_launch<EPI, FORM, true>(p, parts, slab, tail, st) : few_launch<EPI, FORM, false>(p, parts, slab, tail, st);
}
template <int EPI>
int few_run(int form, const GemmParams& p, int parts, float* slab, hipStream_t st, const TailOf<EPI>& tail = {}) {
    static_assert(few::N_FORMS == 5, "forms");
    if constexpr (EPI == QIE_EPI_SWIGLU) {   // (few::choose)
        return form == 1 ? few_one<EPI, 1>(p, parts, slab, tail, st) : few_one<EPI, 2>(p, parts, slab, tail, st);
    } else {
        switch (form) {
            case 0: return few_one<EPI, 0>(p, parts, slab, tail, st);
            case 1: return few_one<EPI, 1>(p, parts, slab, tail, st);
            case 2: return few_one<EPI, 2>(p, parts, slab, tail, st);
            case 3: return few_one<EPI, 3>(p, parts, slab, tail, st);
            default: return few_one<EPI, 4>(p, parts, slab, tail, st);
        }
    }
}
}  // namespace

int gemm_few(const qie_linear_args* a, const GemmParams& p, const QkvTail* tail, hipStream_t st, bool* launched) {
    const bool gated = a->epilogue == QIE_EPI_SWIGLU;
    const few::Plan pl = few::choose(a->M, gated ? 2 * a->N : a->N, a->K, device_cu_count(), gated, a->seg_rows[0] != a->N && (a->seg_rows[0] % 64 || a->seg_rows[1] % 64));
    *launched = pl.form >= 0 && mid::strides_fit(a->ldx, a->ldy);
    if (!*launched) return 0;
    if (tail) return few_run<kEpiQkv>(pl.form, p, 1, nullptr, st, *tail);
    switch (a->epilogue) {
        case QIE_EPI_SWIGLU: return few_run<QIE_EPI_SWIGLU>(pl.form, p, 1, nullptr, st);
        case QIE_EPI_RESIDUAL: return few_run<QIE_EPI_RESIDUAL>(pl.form, p, 1, nullptr, st);
        case QIE_EPI_F32: return few_run<QIE_EPI_F32>(pl.form, p, 1, nullptr, st);
        default: return few_run<QIE_EPI_STORE>(pl.form, p, 1, nullptr, st);
    }
}

int gemm_few_parts(const GemmParams& p, int form, const G8Split& sk, hipStream_t st) { return few_run<kEpiParts>(form, p, sk.splitk, sk.slab, st); }

}  // namespace qie
