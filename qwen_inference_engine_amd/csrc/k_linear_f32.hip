// k_linear_f32.hip — fp32 products of more than a handful of rows for the layered models' fp32 engine.
//
//   Y[m, n] = sum_k A[m, k] W[n, k], plain, per head (batch) or per expert (grp_off: rows by group), on the fp32 matrix cores
//   (v_mfma_f32_16x16x4f32: fp32 products and sums).
//
// The FMA kernel it replaces (k_layered.hip linear_kernel) keeps nothing in flight and fills 32 to 80 of 256 CUs at a few
// hundred rows: 145 to 230 us for 1 to 2 GFLOP.  Here a 64 x 64 tile goes through an LDS-DMA ring of 32-k tiles (128-byte rows,
// as k_gemm_mid.hip), 8 waves as 2 x 2 x 2 K halves, and tiles that do not fill the chip are split over K (slabs summed by the
// last part, gemm8_kernel's protocol).  Bound: the fp32 matrix rate (157 TFLOP/s) or, at few rows, the weights.  us: 275 rows x 1,024 x
// 2,816 230 -> 22, eight experts of some 69 rows (1,024 x 1,408 and 704 x 1,024) 189 and 174 -> 32 and 20.
// Tiles of 32 x 64 (half the row fragments a wave) where rows are few, lf::tile_rows.  (Rings of 5 and 6 slots: no change.)
//   * The order of a sum depends on K alone: K is cut into 1 to 16 segments (a power of two), a wave's segment sums meet in pairs,
//     pairs of pairs and so on, and at last the two K halves.  A workgroup owns an aligned group of segments, one node of that tree,
//     so how many workgroups share a tile (by the rows of the launch and the memory there is for slabs) changes no bit.
#include "gemm_impl.hpp"
#include "gemm_plan.hpp"
#include "k_layered.hpp"

#include <algorithm>

namespace qie {
namespace lay {

namespace lf {
using namespace qie::lf;                   // gemm_plan.hpp
constexpr int SLOTS = 4;
constexpr int slot_bytes(int bm) { return (bm + BN) * BK * 4; }   // A rows, then W rows, 128 B each
}

struct LinF32P {
    LinearP q;
    lf::Plan pl;
    int vec;            // rows of Y take 16-byte stores
    float* slab;        // [tile][part][K half][rows * 64]
    unsigned* cnt;      // [tile], zero at rest
};

// Node `i` (0, 1, 2, ... of its level) of a binary tree of 2^log_n nodes arrives in v; lvl[l] holds a left node that waits for its
// right sibling.  true: it was the last one, v is the tree's root.
template <int L = 0, int FR>
__device__ __forceinline__ bool lf_meet(f32x4 (&v)[FR][2], f32x4 (&lvl)[lf::LEVELS][FR][2], int i, int log_n) {
    if constexpr (L < lf::LEVELS) {
        if (L == log_n) return true;
        if (!((i >> L) & 1)) {
#pragma unroll
            for (int a = 0; a < FR; a++)
#pragma unroll
                for (int b = 0; b < 2; b++) lvl[L][a][b] = v[a][b];
            return false;
        }
#pragma unroll
        for (int a = 0; a < FR; a++)
#pragma unroll
            for (int b = 0; b < 2; b++) v[a][b] = lvl[L][a][b] + v[a][b];
        return lf_meet<L + 1>(v, lvl, i, log_n);
    }
    return true;
}

// FR: fragments of 16 rows a wave; tiles of 32 FR rows
template <int FR>
__global__ __launch_bounds__(512) void linear_f32_kernel(LinF32P p) {
#pragma clang fp contract(off)
    using namespace lf;
    constexpr int BM = 32 * FR, SLOT = slot_bytes(BM), SLAB = slab(BM);
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;
    const int fr = lane & 15, g = lane >> 4;
    const int z = blockIdx.z, nt = blockIdx.x % p.pl.n_nt, part = blockIdx.x / p.pl.n_nt, mt = blockIdx.y;
    int m_lo = 0, m_hi = p.q.M;
    if (p.q.grp_off) {
        m_lo = p.q.grp_off[z];
        m_hi = p.q.grp_off[z + 1];
    }
    const int m0 = m_lo + mt * BM, n0 = nt * BN;
    if (m0 >= m_hi) return;   // block-uniform
    const float* A = p.q.A + (int64_t)z * p.q.sA;
    const float* W = (const float*)p.q.W + (int64_t)z * p.q.sW;
    const int nk_all = p.q.K / BK, log_own = p.pl.log_segs - p.pl.log_parts, parts = 1 << p.pl.log_parts;
    auto seg_at = [&](int seg) { return (int)(((int64_t)seg * nk_all) >> p.pl.log_segs); };   // first k-tile of a segment
    const int seg0 = part << log_own, kb = seg_at(seg0), nk = seg_at((part + 1) << log_own) - kb;

    // LDS-DMA: a wave fills rows 8 wave .. 8 wave + 7 of W, and of A where it has as many
    const bool has_a = FR == 2 || wave < BM / 8;
    const float* src[2];
    {
        const int r = 8 * wave + (lane >> 3), cs = (lane & 7) ^ g8_swz(r);
        const int ar = m0 + r < m_hi ? m0 + r : m_hi - 1;         // rows past the group: its last again, never stored
        const int wr = n0 + r < p.q.N ? n0 + r : p.q.N - 1;
        src[0] = A + (int64_t)ar * p.q.lda + (int64_t)kb * BK + cs * 4;
        src[1] = W + (int64_t)wr * p.q.ldw + (int64_t)kb * BK + ((lane & 7) ^ g8_swz(BM + r)) * 4;
    }
    auto stage = [&](int kt, int slot) {
        unsigned char* dst = smem + slot * SLOT + wave * 1024;
        if (has_a) glds16(src[0] + (int64_t)kt * BK, dst);
        glds16(src[1] + (int64_t)kt * BK, dst + BM * 128);
    };
    f32x4 acc[FR][2], lvl[LEVELS][FR][2];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < FR; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    };
    clear();
    int seg = 0, seg_end = seg_at(seg0 + 1) - kb;
    for (int t = 0; t < SLOTS - 1 && t < nk; t++) stage(t, t);
    int slot = 0, fill = SLOTS - 1;
    for (int t = 0; t < nk; t++) {
        if (t + SLOTS - 1 <= nk && has_a) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (SLOTS - 2)) : "memory");
        else if (t + SLOTS - 1 <= nk) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(SLOTS - 2) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (t + SLOTS - 1 < nk) stage(t + SLOTS - 1, fill);
        const unsigned char* buf = smem + slot * SLOT;
        // this K half: 16 k as four pieces; element e of piece 4 wk + g is k = 4 (4 wk + g) + e in both operands
        f32x4 fa[FR], fb[2];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int row = BM + wn * 32 + j * 16 + fr;
            fb[j] = *reinterpret_cast<const f32x4*>(buf + row * 128 + (((4 * wk + g) ^ g8_swz(row)) * 16));
        }
#pragma unroll
        for (int i = 0; i < FR; i++) {
            const int row = wm * 16 * FR + i * 16 + fr;
            fa[i] = *reinterpret_cast<const f32x4*>(buf + row * 128 + (((4 * wk + g) ^ g8_swz(row)) * 16));
        }
        if (t == seg_end) {   // uniform; a segment is summed: here, while the fragments are on their way
            lf_meet(acc, lvl, seg, log_own);
            clear();
            seg++;
            seg_end = seg_at(seg0 + seg + 1) - kb;
        }
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int i = 0; i < FR; i++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[j][e], fa[i][e], acc[i][j], 0, 0, 0);   // W Aᵀ
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        slot = slot + 1 == SLOTS ? 0 : slot + 1;
        fill = fill + 1 == SLOTS ? 0 : fill + 1;
    }
    lf_meet(acc, lvl, seg, log_own);   // the last segment: acc is this workgroup's node
    if (parts > 1) {
        const int64_t tile = row_tile(p.q.grp_off != nullptr, m0, z, mt, p.pl.n_mt, BM) * p.pl.n_nt + nt;
        const auto rs = __builtin_amdgcn_make_buffer_rsrc(p.slab + ((tile << p.pl.log_parts) + part) * SLAB, (short)0, SLAB * 4, 0x00020000);
#pragma unroll
        for (int i = 0; i < FR; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_g8, acc[i][j]), rs, (((wave * FR + i) * 2 + j) * 64 + lane) * 16, 0, 16);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        int* flag = reinterpret_cast<int*>(smem);
        if (tid == 0) {
            const unsigned old = __hip_atomic_fetch_add(p.cnt + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *flag = old == (unsigned)parts - 1 ? 1 : 0;
        }
        __syncthreads();
        if (*flag == 0) return;   // uniform
        constexpr int QN = 4;     // parts in flight
        for (int q0 = 0; q0 < parts; q0 += QN) {
            f32x4 v[QN][FR][2];
#pragma unroll
            for (int u = 0; u < QN; u++) {
                const int q = q0 + u < parts ? q0 + u : parts - 1;
                const auto rq = __builtin_amdgcn_make_buffer_rsrc(p.slab + ((tile << p.pl.log_parts) + q) * SLAB, (short)0, SLAB * 4, 0x00020000);
#pragma unroll
                for (int i = 0; i < FR; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++)
                        v[u][i][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rq, (((wave * FR + i) * 2 + j) * 64 + lane) * 16, 0, 16));
            }
            // the tree's first two levels here, the others by their waiting nodes
#pragma unroll
            for (int i = 0; i < FR; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const f32x4 lo = v[0][i][j] + v[1][i][j];
                    acc[i][j] = parts == 2 ? lo : lo + (v[2][i][j] + v[3][i][j]);
                }
            if (parts > 2) lf_meet<2>(acc, lvl, q0, p.pl.log_parts);
        }
        if (tid == 0) __hip_atomic_store(p.cnt + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // the two K halves: wave w and w ^ 4 hold the same tile, each keeps one of its two row fragments (FR = 1: column fragments)
    f32x4 res[FR];
    {
        f32x4* ex = reinterpret_cast<f32x4*>(smem);
        auto mine = [&](int j, int half) { return FR == 2 ? acc[half ? FR - 1 : 0][j] : acc[0][half]; };
        __syncthreads();
#pragma unroll
        for (int j = 0; j < FR; j++) {
            ex[(wave * FR + j) * 64 + lane] = wk == 0 ? mine(j, 1) : mine(j, 0);
            res[j] = wk == 0 ? mine(j, 0) : mine(j, 1);
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < FR; j++) {
            const f32x4 o = ex[((wave ^ 4) * FR + j) * 64 + lane];
            res[j] = wk == 0 ? res[j] + o : o + res[j];
        }
    }
    const int m = m0 + wm * 16 * FR + (FR == 2 ? wk * 16 : 0) + fr;
    if (m >= m_hi) return;
    float* Y = p.q.Y + (int64_t)z * p.q.sY + (int64_t)m * p.q.ldy;
#pragma unroll
    for (int j = 0; j < FR; j++) {
        const int n = n0 + wn * 32 + (FR == 2 ? j : wk) * 16 + 4 * g;
        if (p.vec && n + 4 <= p.q.N) {
            *reinterpret_cast<f32x4*>(Y + n) = res[j];
        } else {
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (n + r < p.q.N) Y[n + r] = res[j][r];
        }
    }
}

template <int FR>
static int launch_f32(LinF32P& p, hipStream_t st) {
    constexpr int BM = 32 * FR, SLAB = lf::slab(BM);
    constexpr size_t shm = (size_t)lf::SLOTS * lf::slot_bytes(BM);
    static_assert(shm <= 65536, "linear_f32: default LDS");
    // (grouped: one group may hold every row; the other groups' blocks leave at once)
    p.pl = lf::plan(p.q.M, p.q.N, p.q.K, p.q.batch, p.q.grp_off != nullptr, device_cu_count(), BM);
    if (p.pl.log_parts > 0) {
        G8Split ws{1, nullptr, nullptr};
        const int64_t tiles = p.pl.row_tiles * p.pl.n_nt, slabs = ((tiles << p.pl.log_parts) * SLAB + 65535) / 65536;
        if (g8_workspace(st, (int)slabs, (int)tiles, &ws) != 0) p.pl.log_parts = 0;
        p.slab = ws.slab;
        p.cnt = ws.cnt;
    }
    hipLaunchKernelGGL(linear_f32_kernel<FR>, dim3((unsigned)(p.pl.n_nt << p.pl.log_parts), (unsigned)p.pl.n_mt, (unsigned)p.q.batch), dim3(512), shm, st, p);
    QIE_LAUNCH_CHECK();
    return 0;
}

int linear_f32(const LinearP& q, hipStream_t st, bool* done) {
    using namespace lf;
    const int64_t a16 = (uintptr_t)q.A % 16 + (uintptr_t)q.W % 16;
    *done = !q.round_a && q.M > 16 && (!q.grp_off || q.M > 32) && q.K % BK == 0 && q.lda % 4 == 0 && q.ldw % 4 == 0 && q.sA % 4 == 0 &&
            q.sW % 4 == 0 && a16 == 0;
    if (!*done) return 0;
    LinF32P p{};
    p.q = q;
    p.vec = q.ldy % 4 == 0 && q.sY % 4 == 0 && (uintptr_t)q.Y % 16 == 0;
    return lf::tile_rows(q.M, q.N, q.batch, q.grp_off != nullptr) == 32 ? launch_f32<1>(p, st) : launch_f32<2>(p, st);
}

}  // namespace lay
}  // namespace qie
