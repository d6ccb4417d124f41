// k_decode_bf16.hip — batched decode projections on bf16 weights (2 <= M <= 16 rows).
//
//   Y[M, N] = X[M, K] . W[N, K]^T with the RMSNorm of X in front where it is asked for, and the epilogues of qie_linear.
//
// The weights are all the traffic.  The register-fed skinny kernel (k_gemv.hip) loads its fragments as 16 rows x 64 B and
// waits for them at every step: 4.7 TB/s for Qwen2-7B's gate/up at 4 rows.  Here a workgroup of 8 waves owns whole tiles of
// 16 weight rows, and every wave streams the 128-k chunks of its own share of K (256 contiguous bytes of each row, 4 KB) by
// LDS-DMA through a ring of its own, with no barrier: the loads of R - 1 chunks fly while one is multiplied
// (v_mfma_f32_16x16x32_bf16, D = W Xᵀ, so a lane ends with four neighbouring columns of one row).
//   * X lies in LDS for the whole launch: normed once a workgroup by the waves themselves, under the first chunks' loads, or sent
//     there as it is by LDS-DMA; where M rows of K do not fit (the down projection) its chunks travel through the ring beside the
//     weights'.
//   * Launches of 5 to 15 us feel every instruction and trip to memory ahead of the first product: loads are buffer loads (scalar
//     offsets, no bounds tests), a tile lies in one weight segment so its base is scalar, the first tile's residuals or biases are
//     loaded ahead of the weights, and the wait for X is a counted one.  us before -> with that, Qwen2-7B at 4 rows: QKV 13.2 ->
//     11.1, O 8.8 -> 7.5, gate/up 50.2 -> 48.4; Qwen2-0.5B at 7 rows: QKV 6.4 -> 5.3, O and down 6.5 -> 6.1 a launch.
//   * The 8 partial tiles meet in LDS, one barrier a tile; the wave that sums them and runs the epilogue rotates.
//   * Weights are read with the non-temporal hint (X is not: every workgroup reads it).  Without it they take L2's place from X and
//     from each other: Qwen2-7B's step at 4 rows 3.27 ms -> 2.94, Qwen2-0.5B's at 7 rows 0.93 -> 0.89.
//   * SwiGLU: a tile is 8 gate rows and the same outputs' 8 up rows, met across lane halves.
//   * Gated: the layered models' feed-forward, whose activation is one of fp32 gate and up sums: tiles of 8 + 8 rows as SwiGLU's, behind
//     the tiles of the mixer's rows where one product makes both.  48 launches of 4.7 us fewer in 14 steps of Nukizen's 2k size: 6.52 -> 6.40 ms.
// One workgroup a CU: LDS holds 64 to 128 KB of chunks.  Sums: per wave over its K share in fp32, the shares in wave order (fp32
// operands: 16 sums a wave, met in pairs).
#include "qie_common.hpp"
#include "../../include/qie/qie_ops.h"
#include "k_layered.hpp"

#include <algorithm>
#include <type_traits>

namespace qie {

typedef __bf16 db_bf16x8 __attribute__((ext_vector_type(8)));
typedef float db_f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int db_u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int db_u32x2 __attribute__((ext_vector_type(2)));

namespace db {
constexpr int NW = 8;          // waves
constexpr int CH = 128;        // k of a chunk
constexpr int WCH = 16 * 256;  // bytes of a weight chunk
}

struct DecBfParams {
    const uint16_t* x;
    int64_t ldx;
    const uint16_t* norm_w;
    float eps;
    int numerics;
    const uint16_t* w[3];
    const uint16_t* bias[3];
    int rows[3];               // of the segments (SwiGLU: N, N)
    int t0, t01;               // tiles of segment 0, of segments 0 and 1: a tile lies in one segment
    int K, N, M;
    int n_tiles;
    uint16_t* y;
    int64_t ldy;
    int vec;                   // 8- (fp32: 16-) byte stores
    unsigned long long* keys;
    int64_t key_col0;
    int xstride;               // bytes of a row of the X image (whole 1,024 and 16: 16 rows' same chunk in different banks)
    // kEpiGated
    int act;
    float limit;
    int vec_h;
    uint16_t* h;
    int64_t ldh;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t db_rsrc(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

constexpr int kEpiGated = 5;   // after the QIE_EPI_ values: rows[0] rows as QIE_EPI_F32, then pairs of rows of w[1] and w[2] (lay::GatedP)

// XM: 0 = X in LDS; 8, 16 = X's chunks (of 8 or 16 rows) through the ring.  NV: 16-byte vectors of a row per lane while X is
// normed (K <= 512 NV), 0: not normed, its rows go to LDS as they are; R: ring slots a wave.
// F32: rows of fp32 instead (p.K, p.ldx in 16-bit units; the fp32 epilogue, no norm): a 16-byte piece is 4 k, four
// v_mfma_f32_16x16x4f32 instead of one v_mfma_f32_16x16x32_bf16.  Each of a chunk's 16 instructions has a sum of its own, and
// these and the waves' meet in pairs: a sum is a chain of K / 128 terms at most, not of K / 8 (the Lugipel design at width 1,024,
// decode steps against 64 bits: 4.5e-7 to 5.6e-7 of the logits with one chain a wave, 2.6e-7 to 3.4e-7 so; the column-per-wave kernel 3.4e-7 to 4.2e-7).
template <int EPI, int XM, int NV, int R, bool F32 = false>
__global__ __launch_bounds__(512) void dec_bf16_kernel(DecBfParams p) {
#pragma clang fp contract(off)
    constexpr int SLOT = db::WCH + XM * 256;
    constexpr int IPC = 4 + XM / 4;   // LDS-DMA instructions of a chunk (4 rows of 256 B each)
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, g = lane >> 4;
    unsigned char* ring = smem + wave * (R * SLOT);
    const int M = p.M, K = p.K;
    // partial tiles [2][NW][RS]: all 64 lanes' quads, or those of X rows 0 .. 7
    const int RS = M <= 8 ? 32 : 64, rl = M <= 8 ? g * 8 + (fr & 7) : lane;
    db_f32x4* red = reinterpret_cast<db_f32x4*>(smem + db::NW * R * SLOT);
    unsigned char* xs = smem + db::NW * R * SLOT + 2 * db::NW * RS * 16;
    const int chunks = K / db::CH;
    const int c0 = wave * chunks / db::NW, cnt = (wave + 1) * chunks / db::NW - c0;   // this wave's share of K
    const int T = p.n_tiles, G = gridDim.x;
    const int mine = ((int)blockIdx.x < T) ? (T - 1 - (int)blockIdx.x) / G + 1 : 0;
    const int items = mine * cnt;   // (tile, chunk) in order

    // ---- X rows for the norm (or the copy), loaded ahead of the first weight chunks: P waves a row (8, 4, 2 rows at a time), so
    // that few rows keep every wave busy.  (Buffer loads throughout: a load is one instruction with its offset in a scalar register,
    // and what lies past K reads zeros.  With 64-bit addresses and a bounds test a lane the prologue was ~2,000 instructions.)
    const int P = M <= 2 ? 4 : M <= 4 ? 2 : 1, sub = wave % P;
    db_u32x4 xv[NV ? NV : 1], nv[NV ? NV : 1];
    auto load_row = [&](int m) {
        const auto rx = db_rsrc(p.x + (int64_t)m * p.ldx, (uint32_t)K * 2), rn = db_rsrc(p.norm_w, (uint32_t)K * 2);
#pragma unroll
        for (int v = 0; v < NV; v++) {
            if ((v * P + sub) * 512 >= K) break;   // uniform
            xv[v] = __builtin_amdgcn_raw_buffer_load_b128(rx, lane * 16, (v * P + sub) * 1024, 0);
            nv[v] = __builtin_amdgcn_raw_buffer_load_b128(rn, lane * 16, (v * P + sub) * 1024, 0);
        }
    };
    if constexpr (XM == 0 && NV > 0) {
        if (wave / P < M) load_row(wave / P);
    } else if constexpr (XM == 0) {
        for (int m = wave; m < M; m += db::NW) {
            const auto rx = db_rsrc(p.x + (int64_t)m * p.ldx, (uint32_t)K * 2);
            for (int c = 0; c * 512 < K; c++) buffer_lds16(rx, xs + m * p.xstride + c * 1024, lane * 16, c * 1024);
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    // ---- tiles: segment, first row in it, rows left, first column (uniform)
    struct Tile {
        int seg, row0, left, col;
    };
    auto tile_at = [&](int tile) {
        Tile t;
        if constexpr (EPI == QIE_EPI_SWIGLU) {
            t.seg = 0;
            t.row0 = t.col = tile * 8;
        } else if constexpr (EPI == kEpiGated) {
            t.seg = tile < p.t0 ? 0 : 1;
            t.row0 = t.col = t.seg == 0 ? tile * 16 : (tile - p.t0) * 8;
        } else {
            t.seg = tile < p.t0 ? 0 : tile < p.t01 ? 1 : 2;
            t.row0 = (tile - (t.seg == 0 ? 0 : t.seg == 1 ? p.t0 : p.t01)) * 16;
            t.col = t.row0 + (t.seg == 0 ? 0 : t.seg == 1 ? p.rows[0] : p.rows[0] + p.rows[1]);
        }
        t.left = (t.seg == 0 ? p.rows[0] : t.seg == 1 ? p.rows[1] : p.rows[2]) - t.row0;
        return t;
    };
    // the epilogue's operands: old values (whole quads), or biases.  The first tile's are loaded by the wave that will need them ahead of
    // its chunks: behind the reduction they cost another trip to memory, and most launches have one tile a block.
    db_u32x2 old = {0u, 0u};
    uint32_t bias[4] = {0u, 0u, 0u, 0u};
    auto load_old = [&](const Tile& t, bool on) {
        const auto ry = db_rsrc(p.y, on && p.vec ? (uint32_t)(((int64_t)(M - 1) * p.ldy + p.N) * 2) : 0u);
        old = __builtin_amdgcn_raw_buffer_load_b64(ry, (int)((fr * (int)p.ldy + t.col + 4 * g) * 2), 0, 0);
    };
    auto load_bias = [&](const Tile& t, bool on) {
        const uint16_t* b = t.seg == 0 ? p.bias[0] : t.seg == 1 ? p.bias[1] : p.bias[2];
        const auto rb = db_rsrc(b ? b : p.x, b && on ? (uint32_t)(t.row0 + t.left) * 2 : 0u);   // none: zeros
#pragma unroll
        for (int r = 0; r < 4; r++) bias[r] = __builtin_amdgcn_raw_buffer_load_b16(rb, (t.row0 + 4 * g + r) * 2, 0, 0);
    };
    {
        const Tile t = tile_at(mine > 0 ? (int)blockIdx.x : 0);
        if constexpr (EPI == QIE_EPI_RESIDUAL) load_old(t, wave == 0);
        if constexpr (EPI == QIE_EPI_STORE) load_bias(t, wave == 0);
        __builtin_amdgcn_sched_barrier(0);
    }

    // ---- the weight stream: lane -> row 4 i + (lane >> 4) of the tile, LDS piece lane & 15 of its 256 B, which holds the
    // source's piece (lane & 15) ^ row (the fragment reads below are then free of bank conflicts)
    uint32_t wsrc[4], xsrc[XM ? XM / 4 : 1];
    const uint32_t xbytes = (uint32_t)(((int64_t)(M - 1) * p.ldx + K) * 2);
    if constexpr (XM != 0) {
#pragma unroll
        for (int i = 0; i < XM / 4; i++) {
            const int m = 4 * i + (lane >> 4);
            xsrc[i] = (uint32_t)((m < M ? m : M - 1) * (int)p.ldx * 2 + ((lane & 15) ^ m) * 16);
        }
    }
    const uint16_t *wb0 = nullptr, *wb1 = nullptr;   // the tile's first row (SwiGLU: of gate and up)
    uint32_t wbytes = 0;
    auto aim = [&](int tile) {
        const Tile t = tile_at(tile);
        const int64_t at = (int64_t)t.row0 * K;
        wb0 = (t.seg == 0 ? p.w[0] : t.seg == 1 ? p.w[1] : p.w[2]) + at;
        if constexpr (EPI == QIE_EPI_SWIGLU) wb1 = p.w[1] + at;
        if constexpr (EPI == kEpiGated) wb1 = t.seg == 0 ? wb0 : p.w[2] + at;
        const int TR = EPI == QIE_EPI_SWIGLU || (EPI == kEpiGated && t.seg == 1) ? 8 : 16;
        wbytes = (uint32_t)(t.left < TR ? t.left : TR) * (uint32_t)K * 2;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int row = 4 * i + (lane >> 4), r = row & (TR - 1);
            wsrc[i] = (uint32_t)((r < t.left ? r : t.left - 1) * K * 2 + ((lane & 15) ^ row) * 16);
        }
    };
    int n_tile = blockIdx.x, n_c = 0, n_slot = 0;   // the next chunk to ask for
    auto issue = [&](bool on) {   // off: nothing is read
        unsigned char* dst = ring + n_slot * SLOT;
        const uint32_t k = (uint32_t)(c0 + n_c) * 256;
        const auto r0 = db_rsrc(wb0, on ? wbytes : 0u), r1 = EPI == QIE_EPI_SWIGLU || EPI == kEpiGated ? db_rsrc(wb1, on ? wbytes : 0u) : r0;
#pragma unroll
        for (int i = 0; i < 4; i++) buffer_lds16<true>(i < 2 ? r0 : r1, dst + i * 1024, wsrc[i], k);
        if constexpr (XM != 0) {
#pragma unroll
            for (int i = 0; i < XM / 4; i++) buffer_lds16(db_rsrc(p.x, on ? xbytes : 0u), dst + db::WCH + i * 1024, xsrc[i], k);
        }
        n_slot = n_slot + 1 == R ? 0 : n_slot + 1;
        if (++n_c == cnt) {
            n_c = 0;
            n_tile += G;
            aim(n_tile < T ? n_tile : T - 1);
        }
    };
    aim(n_tile);
    // R chunks whatever there are, so that the wait for X is a counted one that leaves them in flight
#pragma unroll
    for (int i = 0; i < R; i++) issue(i < items);
    __builtin_amdgcn_sched_barrier(0);

    if constexpr (XM == 0) {
        if constexpr (NV > 0) {   // M <= 8: one pass
            // The sum of squares in qie_rmsnorm's order, whatever P is: a row's 512-k pieces go to four sums in turn, each over a wave.
            const int m = wave / P;
            float* ssq = reinterpret_cast<float*>(red);   // [row][4]
            auto squares = [&](auto pc) {
                constexpr int PP = decltype(pc)::value, S = 4 / PP;   // this wave's sums: pieces v PP + sub, v = j, j + S, ...
                float ss[S] = {};
#pragma unroll
                for (int v = 0; v < (NV + PP - 1) / PP; v++) {
                    if ((v * PP + sub) * 512 >= K) break;
                    const uint32_t e[4] = {xv[v].x, xv[v].y, xv[v].z, xv[v].w};
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const float a = bf_lo(e[j]), b = bf_hi(e[j]);
                        ss[v % S] += a * a + b * b;
                    }
                }
                // wave_sum of all of them at once: a lane exchange takes two values, and row r of 16 lanes ends with sum r
#pragma unroll
                for (int j = 0; j < S; j++) ss[j] = group_sum<16>(ss[j]);
                float t;
                if constexpr (S == 1) {
                    t = xor32_sum(xor16_sum(ss[0]));
                } else {
                    lane_swap<16>(ss[0], ss[1]);
                    t = ss[0] + ss[1];
                    if constexpr (S == 4) {
                        lane_swap<16>(ss[2], ss[3]);
                        float u = ss[2] + ss[3];
                        lane_swap<32>(t, u);
                        t = t + u;
                    } else {
                        t = xor32_sum(t);
                    }
                }
                if ((lane & 15) == 0 && lane < 16 * S) ssq[m * 4 + (lane >> 4) * PP + sub] = t;
            };
            if (P == 1) squares(std::integral_constant<int, 1>{});
            else if (P == 2) squares(std::integral_constant<int, 2>{});
            else squares(std::integral_constant<int, 4>{});
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (not __syncthreads: the chunks in flight stay there)
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            const float tot = ssq[m * 4] + ssq[m * 4 + 1] + ssq[m * 4 + 2] + ssq[m * 4 + 3];
            const float rms = sqrtf((tot / (float)K) + p.eps), inv = 1.0f / rms, rr = rms < INFINITY ? rms : 0.f;
            auto apply = [&](auto hf) {
                constexpr bool HF = decltype(hf)::value;
#pragma unroll
                for (int v = 0; v < NV; v++) {
                    if ((v * P + sub) * 512 >= K) break;
                    xv[v].x = rms_pair<HF>(xv[v].x, nv[v].x, rr, inv);
                    xv[v].y = rms_pair<HF>(xv[v].y, nv[v].y, rr, inv);
                    xv[v].z = rms_pair<HF>(xv[v].z, nv[v].z, rr, inv);
                    xv[v].w = rms_pair<HF>(xv[v].w, nv[v].w, rr, inv);
                }
            };
            if (m < M) {
                if (p.numerics == QIE_NUMERICS_HF) apply(std::true_type{});
                else apply(std::false_type{});
#pragma unroll
                for (int v = 0; v < NV; v++) {
                    if ((v * P + sub) * 512 >= K) break;
                    *reinterpret_cast<db_u32x4*>(xs + m * p.xstride + (v * P + sub) * 1024 + lane * 16) = xv[v];
                }
            }
        } else {
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(IPC * R) : "memory");   // X is there; the chunks fly on
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    }

    // (the wait for them belongs here, not into the loop of counted waits)
    asm volatile("" : "+v"(old), "+v"(bias[0]), "+v"(bias[1]), "+v"(bias[2]), "+v"(bias[3]));
    const int arow = fr < M ? fr : M - 1;   // rows past M: copies of row M - 1, never stored
    unsigned long long kbest = 0ull;
    int done = 0, slot = 0;
    for (int it = 0; it < mine; it++) {
        const int tile = blockIdx.x + it * G;
        db_f32x4 acc = {0.f, 0.f, 0.f, 0.f}, af[F32 ? 16 : 1];
        if constexpr (F32) {
#pragma unroll
            for (int i = 0; i < 16; i++) af[i] = acc;
        }
        for (int c = 0; c < cnt; c++) {
            // the oldest chunk has landed: R - 1 younger ones may fly (fewer at the end of the stream)
            if (done + R <= items) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(IPC * (R - 1)) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            const unsigned char* buf = ring + slot * SLOT;
            db_bf16x8 wf[4], xf[4];
#pragma unroll
            for (int s = 0; s < 4; s++) {
                wf[s] = *reinterpret_cast<const db_bf16x8*>(buf + fr * 256 + (((4 * s + g) ^ fr) * 16));
                if constexpr (XM == 0)
                    xf[s] = *reinterpret_cast<const db_bf16x8*>(xs + arow * p.xstride + (c0 + c) * 256 + (4 * s + g) * 16);
                else
                    xf[s] = *reinterpret_cast<const db_bf16x8*>(buf + db::WCH + (fr & (XM - 1)) * 256 + (((4 * s + g) ^ (fr & (XM - 1))) * 16));
            }
#pragma unroll
            for (int s = 0; s < 4; s++) {
                if constexpr (F32) {
                    const db_f32x4 a = __builtin_bit_cast(db_f32x4, wf[s]), b = __builtin_bit_cast(db_f32x4, xf[s]);
#pragma unroll
                    for (int e = 0; e < 4; e++) af[4 * s + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], af[4 * s + e], 0, 0, 0);
                } else {
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[s], xf[s], acc, 0, 0, 0);
                }
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the slot's reads are done
            __builtin_amdgcn_sched_barrier(0);
            if (done + R < items) issue(true);
            done++;
            slot = slot + 1 == R ? 0 : slot + 1;
        }
        if constexpr (F32) {
#pragma unroll
            for (int o = 8; o >= 1; o >>= 1)
#pragma unroll
                for (int i = 0; i < o; i++) af[i] = af[i] + af[i + o];
            acc = af[0];
        }
        if (fr < 8 || M > 8) red[((it & 1) * db::NW + wave) * RS + rl] = acc;
        // one barrier a tile: a slot of `red` is written again two tiles on, behind the next tile's barrier, which the summing
        // wave reaches only after its reads.  (No vmcnt wait: the ring's loads stay in flight.)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (wave != it % db::NW) continue;   // wave-uniform
        db_f32x4 v = red[(it & 1) * db::NW * RS + rl];
        if constexpr (F32) {
            db_f32x4 u[db::NW];
#pragma unroll
            for (int w = 0; w < db::NW; w++) u[w] = red[((it & 1) * db::NW + w) * RS + rl];
            v = ((u[0] + u[1]) + (u[2] + u[3])) + ((u[4] + u[5]) + (u[6] + u[7]));
        } else {
#pragma unroll
            for (int w = 1; w < db::NW; w++) v = v + red[((it & 1) * db::NW + w) * RS + rl];
        }
        const Tile t = tile_at(tile);
        // lane: row m = fr of X, columns 4 g .. 4 g + 3 of the tile (SwiGLU: g = 0, 1 gate, g = 2, 3 the same outputs' up)
        const int m = fr;
        if constexpr (EPI == QIE_EPI_SWIGLU) {
            float h[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float a = v[r], b = v[r];
                lane_swap<32>(a, b);   // lanes 0..31: a = own (gate), b = lane + 32's (up)
                const float gg = rbf(a), uu = rbf(b);
                h[r] = uu * rbf(gg * (1.0f / (1.0f + expf(-gg))));
            }
            const int64_t col = t.col + 4 * g;
            if (g < 2 && m < M) {
                uint16_t* dst = p.y + (int64_t)m * p.ldy + col;
                if (p.vec && col + 4 <= p.N) {
                    *reinterpret_cast<uint2*>(dst) = make_uint2(pack2(h[0], h[1]), pack2(h[2], h[3]));
                } else {
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (col + r < p.N) dst[r] = f2bf(h[r]);
                }
            }
        } else if (EPI == kEpiGated && t.seg == 1) {
            float h[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float a = v[r], b = v[r];
                lane_swap<32>(a, b);   // as SwiGLU's
                h[r] = lay::gated_act(a, b, p.act, p.limit);
            }
            const int64_t col = t.col + 4 * g;
            if (g < 2 && m < M) {
                uint16_t* dst = p.h + (int64_t)m * p.ldh + col;
                if (p.vec_h && col + 4 <= p.rows[1]) {
                    *reinterpret_cast<uint2*>(dst) = make_uint2(pack2(h[0], h[1]), pack2(h[2], h[3]));
                } else {
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (col + r < p.rows[1]) dst[r] = f2bf(h[r]);
                }
            }
        } else if (m < M) {
            const int64_t col = t.col + 4 * g, end = t.col + t.left;   // the segment's end
            const bool whole = p.vec && t.col % 4 == 0 && col + 4 <= end;
            if constexpr (EPI == QIE_EPI_F32 || EPI == kEpiGated) {
                float* dst = reinterpret_cast<float*>(p.y) + (int64_t)m * p.ldy + col;
                if (whole) {
                    *reinterpret_cast<db_f32x4*>(dst) = v;
                } else {
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (col + r < end) dst[r] = v[r];
                }
            } else {
                uint16_t* dst = p.y + (int64_t)m * p.ldy + col;
                float o[4];
                if constexpr (EPI == QIE_EPI_RESIDUAL) {
                    if (whole) {
                        if (it > 0) {
                            const uint2 x = *reinterpret_cast<const uint2*>(dst);
                            old = db_u32x2{x.x, x.y};
                        }
                        o[0] = bf_lo(old.x);
                        o[1] = bf_hi(old.x);
                        o[2] = bf_lo(old.y);
                        o[3] = bf_hi(old.y);
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; r++) o[r] = col + r < end ? bf2f(dst[r]) : 0.f;
                    }
#pragma unroll
                    for (int r = 0; r < 4; r++) o[r] += rbf(v[r]);
                } else {
                    if (it > 0) load_bias(t, true);
#pragma unroll
                    for (int r = 0; r < 4; r++) o[r] = v[r] + bf2f((uint16_t)bias[r]);
                }
                const uint32_t lo = pack2(o[0], o[1]), hi = pack2(o[2], o[3]);
                if (whole) {
                    *reinterpret_cast<uint2*>(dst) = make_uint2(lo, hi);
                } else {
                    const uint16_t q[4] = {(uint16_t)lo, (uint16_t)(lo >> 16), (uint16_t)hi, (uint16_t)(hi >> 16)};
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (col + r < end) dst[r] = q[r];
                }
                if (EPI == QIE_EPI_STORE && p.keys) {
                    const uint32_t q[4] = {lo & 0xffffu, lo >> 16, hi & 0xffffu, hi >> 16};
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        if (col + r >= end) continue;
                        const unsigned long long kk = sel_key(bf2f(q[r]), (uint32_t)(col + r + p.key_col0));
                        kbest = kk > kbest ? kk : kbest;
                    }
                }
            }
        }
    }
    if (EPI == QIE_EPI_STORE && p.keys) {   // the best key of every row: over the lanes and waves, then one atomic a workgroup
        __syncthreads();
        unsigned long long* kb = reinterpret_cast<unsigned long long*>(red);
        kb[wave * 64 + lane] = kbest;
        __syncthreads();
        if (tid < M) {
            unsigned long long b = 0ull;
            for (int w = 0; w < db::NW; w++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const unsigned long long k = kb[w * 64 + q * 16 + tid];
                    b = k > b ? k : b;
                }
            if (b) atomicMax(p.keys + tid, b);
        }
    }
}

// ---------------------------------------------------------------- dispatch
namespace {
constexpr int64_t kDbLds = 160 * 1024;

// X in LDS beside a ring of R slots a wave
int64_t db_red_bytes(int64_t M) { return 2 * db::NW * (M <= 8 ? 512 : 1024); }
int64_t db_image_bytes(int64_t M, int64_t K, int R) { return db::NW * R * db::WCH + db_red_bytes(M) + M * ((K + 511) / 512 * 1024 + 16); }

struct DbPlan {
    int xm, nv, r;
    size_t lds;
};
// Plain rows where the skinny kernel stays ahead, at fewer than 8 rows: its waves divide K of 512, 1,024 and 2,048 without a rest, and
// here half of them have no chunk at 512.  us, skinny | this one, at 2 and 4 rows: 512 x 8,192 gated 6.1 6.9 | 7.9 7.9, 512 x 2,048
// 3.4 3.5 | 3.7 3.8, 1,024 x 8,192 gated 9.1 9.7 | 10.6 10.8, 2,048 x 8,192 9.3 9.7 | 11.2 11.7, 2,048 x 48,000 37.0 39.3 | 41.6 42.4;
// but 512 x 14,336 8.7 9.1 | 7.0 7.1, 640 x 8,192 6.3 6.5 | 5.5 5.6, 2,176 x 8,192 11.3 11.8 | 9.9 9.7, and fp32 outputs (layered
// models) 2,048 x 14,336 15.9 15.4 | 14.4 14.6.  With a norm the skinny kernel needs another launch.
bool db_skinny_ahead(const qie_linear_args* a) {
    if (a->norm_w || a->M >= 8) return false;
    const bool gated = a->epilogue == QIE_EPI_SWIGLU;
    const int64_t rows = gated ? 2 * a->N : a->N;
    if (a->K == 512) return gated || rows <= 8192;
    return (a->K == 1024 || a->K == 2048) && rows >= 8192 && a->epilogue != QIE_EPI_F32;
}
bool db_plan(const qie_linear_args* a, DbPlan* out) {
    if (dev_env("QIE_DEC_BF16", 1) == 0) return false;
    if ((a->flags & QIE_LINEAR_FP8) || a->M < 2 || a->M > 16 || a->K % db::CH != 0 || a->K / db::CH < db::NW / 2) return false;
    if (a->K >= 1 << 26 || a->M * a->ldx >= 1 << 30 || a->M * a->ldy >= 1 << 29) return false;   // 32-bit offsets
    if (a->norm_w && (a->M > db::NW || ((uintptr_t)a->norm_w) % 16 != 0)) return false;
    if (db_skinny_ahead(a)) return false;
    if (a->K <= 5120) {
        // chunks that a wave of the busiest block streams: a slot beyond them is issued for nothing
        const int64_t cus = device_cu_count(), tiles = a->epilogue == QIE_EPI_SWIGLU ? (a->N + 7) / 8 : (a->N + 15) / 16 + 2;
        const int64_t items = (tiles + cus - 1) / cus * ((a->K / db::CH + db::NW - 1) / db::NW);
        for (int r = (int)std::max<int64_t>(2, std::min<int64_t>(4, items)); r >= 2; r--)
            if (db_image_bytes(a->M, a->K, r) <= kDbLds) {
                *out = {0, !a->norm_w ? 0 : a->K <= 1024 ? 2 : a->K <= 2048 ? 4 : a->K <= 3584 ? 7 : 10, r, (size_t)db_image_bytes(a->M, a->K, r)};
                return true;
            }
    }
    if (a->norm_w) return false;
    const int xm = a->M <= 8 ? 8 : 16;
    *out = {xm, 0, 2, (size_t)(db::NW * 2 * (db::WCH + xm * 256) + db_red_bytes(a->M))};
    return true;
}

template <int EPI, int XM, int NV, int R, bool F32 = false>
int db_launch(const DecBfParams& p, size_t lds, hipStream_t st) {
    const void* fn = (const void*)dec_bf16_kernel<EPI, XM, NV, R, F32>;
    static bool raised = false;
    if (!raised) {
        QIE_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kDbLds));
        raised = true;
    }
    const int grid = std::max(1, std::min(p.n_tiles, (int)device_cu_count()));
    hipLaunchKernelGGL((dec_bf16_kernel<EPI, XM, NV, R, F32>), dim3((unsigned)grid), dim3(512), lds, st, p);
    QIE_LAUNCH_CHECK();
    return 0;
}
template <int EPI, int R>
int db_launch_nv(const DecBfParams& p, const DbPlan& pl, hipStream_t st) {
    switch (pl.nv) {
        case 0: return db_launch<EPI, 0, 0, R>(p, pl.lds, st);
        case 2: return db_launch<EPI, 0, 2, R>(p, pl.lds, st);
        case 4: return db_launch<EPI, 0, 4, R>(p, pl.lds, st);
        case 7: return db_launch<EPI, 0, 7, R>(p, pl.lds, st);
        default: return db_launch<EPI, 0, 10, R>(p, pl.lds, st);
    }
}
template <int EPI>
int db_launch_plan(const DecBfParams& p, const DbPlan& pl, hipStream_t st) {
    if (pl.xm == 8) return db_launch<EPI, 8, 0, 2>(p, pl.lds, st);
    if (pl.xm == 16) return db_launch<EPI, 16, 0, 2>(p, pl.lds, st);
    if (pl.r == 4) return db_launch_nv<EPI, 4>(p, pl, st);
    if (pl.r == 3) return db_launch_nv<EPI, 3>(p, pl, st);
    return db_launch_nv<EPI, 2>(p, pl, st);
}
}  // namespace

// whether dec_bf16_linear takes this projection as it stands, its norm included
bool dec_bf16_applies(const qie_linear_args* a) {
    DbPlan pl;
    return db_plan(a, &pl);
}

int dec_bf16_linear(const qie_linear_args* a, hipStream_t st, bool* done) {
    DbPlan pl;
    *done = db_plan(a, &pl);
    if (!*done) return 0;
    DecBfParams p{};
    p.x = (const uint16_t*)a->x;
    p.ldx = a->ldx;
    p.norm_w = (const uint16_t*)a->norm_w;
    p.eps = a->norm_eps;
    p.numerics = a->numerics;
    for (int i = 0; i < 3; i++) {
        p.w[i] = (const uint16_t*)a->w[i];
        p.bias[i] = (const uint16_t*)a->bias[i];
    }
    for (int i = 0; i < 3; i++) p.rows[i] = (int)(a->epilogue == QIE_EPI_SWIGLU ? a->N : a->seg_rows[i]);
    p.t0 = (p.rows[0] + 15) / 16;
    p.t01 = p.t0 + (p.rows[1] + 15) / 16;
    p.K = (int)a->K;
    p.N = (int)a->N;
    p.M = (int)a->M;
    p.n_tiles = a->epilogue == QIE_EPI_SWIGLU ? (p.N + 7) / 8 : p.t01 + (p.rows[2] + 15) / 16;
    p.y = (uint16_t*)a->y;
    p.ldy = a->ldy;
    p.vec = a->ldy % 4 == 0 && ((uintptr_t)a->y) % (a->epilogue == QIE_EPI_F32 ? 16 : 8) == 0;
    p.keys = (unsigned long long*)a->argmax_keys;
    p.key_col0 = a->key_col0;
    p.xstride = (p.K + 511) / 512 * 1024 + 16;
    switch (a->epilogue) {
        case QIE_EPI_SWIGLU: return db_launch_plan<QIE_EPI_SWIGLU>(p, pl, st);
        case QIE_EPI_RESIDUAL: return db_launch_plan<QIE_EPI_RESIDUAL>(p, pl, st);
        case QIE_EPI_F32: return db_launch_plan<QIE_EPI_F32>(p, pl, st);
        default: return db_launch_plan<QIE_EPI_STORE>(p, pl, st);
    }
}

// lay::GatedP for 2 to 16 rows; *done false: not its shape (the sums are those of qie_linear's fp32 product, which comes to the same kernel)
int dec_bf16_gated(const lay::GatedP& q, hipStream_t st, bool* done) {
    qie_linear_args a{};
    a.x = q.x; a.ldx = q.K;
    a.w[0] = q.w; a.seg_rows[0] = a.N = (int64_t)q.plain + 2 * (int64_t)q.ff;
    a.M = q.M; a.K = q.K;
    a.y = q.y; a.ldy = q.ldy;
    a.epilogue = QIE_EPI_F32;
    DbPlan pl;
    *done = q.ff > 0 && (((uintptr_t)q.x | (uintptr_t)q.w) % 16) == 0 && (int64_t)q.M * q.ldh < (int64_t)1 << 29 && db_plan(&a, &pl);
    if (!*done) return 0;
    DecBfParams p{};
    p.x = q.x;
    p.ldx = q.K;
    p.w[0] = (const uint16_t*)q.w;
    p.w[1] = p.w[0] + (int64_t)q.plain * q.K;
    p.w[2] = p.w[1] + (int64_t)q.ff * q.K;
    p.rows[0] = q.plain;
    p.rows[1] = p.rows[2] = q.ff;
    p.t0 = (q.plain + 15) / 16;
    p.n_tiles = p.t0 + (q.ff + 7) / 8;
    p.K = q.K;
    p.N = q.plain;
    p.M = q.M;
    p.y = (uint16_t*)q.y;
    p.ldy = q.ldy;
    p.vec = q.ldy % 4 == 0 && ((uintptr_t)q.y) % 16 == 0;
    p.xstride = (p.K + 511) / 512 * 1024 + 16;
    p.act = q.act;
    p.limit = q.limit;
    p.vec_h = q.ldh % 4 == 0 && ((uintptr_t)q.h) % 8 == 0;
    p.h = q.h;
    p.ldh = q.ldh;
    constexpr int E = kEpiGated;
    if (pl.xm == 8) return db_launch<E, 8, 0, 2>(p, pl.lds, st);
    if (pl.xm == 16) return db_launch<E, 16, 0, 2>(p, pl.lds, st);
    if (pl.r == 4) return db_launch<E, 0, 0, 4>(p, pl.lds, st);
    if (pl.r == 3) return db_launch<E, 0, 0, 3>(p, pl.lds, st);
    return db_launch<E, 0, 0, 2>(p, pl.lds, st);
}

// y = X W^T in fp32 for up to 16 rows (lay::linear's plain form): *done false: not its shape
int dec_f32_linear(const lay::LinearP& q, hipStream_t st, bool* done) {
    *done = q.batch == 1 && !q.grp_off && !q.round_a && q.M <= 16 && q.K % 64 == 0 && q.K >= 256 && q.K < 1 << 25 && q.ldw == q.K && q.lda % 4 == 0 &&
            (int64_t)q.M * q.lda < (int64_t)1 << 29 && (int64_t)q.M * q.ldy < (int64_t)1 << 29 && (((uintptr_t)q.A | (uintptr_t)q.W) % 16) == 0;
    if (!*done) return 0;
    DecBfParams p{};
    p.x = (const uint16_t*)q.A;
    p.ldx = q.lda * 2;
    p.w[0] = (const uint16_t*)q.W;
    p.rows[0] = q.N;
    p.t0 = p.t01 = (q.N + 15) / 16;
    p.K = q.K * 2;
    p.N = q.N;
    p.M = q.M;
    p.n_tiles = p.t0;
    p.y = (uint16_t*)q.Y;
    p.ldy = q.ldy;
    p.vec = q.ldy % 4 == 0 && ((uintptr_t)q.Y) % 16 == 0;
    p.xstride = (p.K + 511) / 512 * 1024 + 16;
    constexpr int E = QIE_EPI_F32;
    if (p.K <= 5120 && db_image_bytes(p.M, p.K, 2) <= kDbLds) return db_launch<E, 0, 0, 2, true>(p, (size_t)db_image_bytes(p.M, p.K, 2), st);
    const int xm = p.M <= 8 ? 8 : 16;
    const size_t lds = (size_t)(db::NW * 2 * (db::WCH + xm * 256) + db_red_bytes(p.M));
    return xm == 8 ? db_launch<E, 8, 0, 2, true>(p, lds, st) : db_launch<E, 16, 0, 2, true>(p, lds, st);
}

}  // namespace qie
