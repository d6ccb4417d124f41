// gemm_impl.hpp — what the prefill GEMMs share (k_gemm.hip, k_gemm_mid.hip): operands, LDS-DMA, the split-K workspace.
#pragma once

#include <type_traits>

#include "qie_common.hpp"
#include "../../include/qie/qie_ops.h"
#include "split_pool.hpp"

namespace qie {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// What follows a QKV projection of prompts laid end to end, each from position 0 on, without q / k norms and with rotary pairs
// (2 i, 2 i + 1): q and k turned, q to its rows, k and v to the cache (qkv_post_kernel's results)
struct QkvTail {
    uint16_t* q;             // [M][qd]
    uint16_t *k, *v;         // the layer's first run
    const float* turns;      // [position][hd / 2][cos, sin]
    int len;                 // rows of a prompt
    int qd, kd;              // columns of q, of k and of v
    int hd_log2;
    KvMap km;
};
constexpr int kEpiQkv = 4;   // the epilogue that does this: k_gemm.hip's 256x256 kernel and k_gemm_mid.hip's have it
constexpr int kEpiParts = 6;   // k_gemm_mid.hip, k_gemm_few.hip: every part of K stores its own sums, fp32 rows [part][M][N], for k_sum_norm.hip
// The last argument of kernels with an epilogue EPI.  As part of every kernel's it moved what lies behind it (the grid's size) to a further line
// of the argument segment: 0.3 us in each launch.
struct NoTail {};
template <int EPI>
using TailOf = std::conditional_t<EPI == kEpiQkv, QkvTail, NoTail>;

struct GemmParams {
    const uint16_t* A;
    int64_t lda;
    const uint16_t* w0;
    const uint16_t* w1;
    const uint16_t* w2;
    const uint16_t* b0;
    const uint16_t* b1;
    const uint16_t* b2;
    int64_t n0, n01;
    int64_t M, K, N;     // N = output columns
    int64_t wrows;       // total weight rows addressable (for clamping)
    uint16_t* C;
    int64_t ldc;
    int vec = 0;         // rows of C take 4-element vector stores
};

__device__ __forceinline__ void glds16(const void* src, void* lds) {
    __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) void*)(src),
                                     (__attribute__((address_space(3))) void*)(lds), 16, 0, 0);
}

// chunk swizzle of 128-B LDS rows: the 16-B chunk c of row r sits at c ^ g8_swz(r)
__device__ __forceinline__ int g8_swz(int r) { return (r >> 1) & 7; }

// ---------------------------------------------------------------- epilogues of four columns a lane
// dst: C at the first of them; `left` columns of the row from there on, the others are not stored.

__device__ __forceinline__ void store_quad(uint16_t* dst, const float (&v)[4], bool vec, int64_t left) {
    if (vec && left >= 4) {
        *reinterpret_cast<uint2*>(dst) = make_uint2(pack2(v[0], v[1]), pack2(v[2], v[3]));
    } else {
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (r < left) dst[r] = f2bf(v[r]);
    }
}
__device__ __forceinline__ void store_quad_f32(float* dst, f32x4 v, bool vec, int64_t left) {
    if (vec && left >= 4) {
        *reinterpret_cast<f32x4*>(dst) = v;
    } else {
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (r < left) dst[r] = v[r];
    }
}
// residual: C = bf16(x + bf16(v)), x what quad_before read there
__device__ __forceinline__ uint2 quad_before(const uint16_t* src, bool vec, int64_t left) {
    if (vec && left >= 4) return *reinterpret_cast<const uint2*>(src);
    uint32_t h[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int r = 0; r < 4; r++)
        if (r < left) h[r] = src[r];
    return make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
}
__device__ __forceinline__ void sum_quad(uint2 x, f32x4 v, float (&o)[4]) {
    o[0] = bf_lo(x.x) + rbf(v[0]);
    o[1] = bf_hi(x.x) + rbf(v[1]);
    o[2] = bf_lo(x.y) + rbf(v[2]);
    o[3] = bf_hi(x.y) + rbf(v[3]);
}
__device__ __forceinline__ void add_quad(uint16_t* dst, uint2 x, f32x4 v, bool vec, int64_t left) {
    float o[4];
    sum_quad(x, v, o);
    store_quad(dst, o, vec, left);
}
// biases of columns col .. col + 3 (zero where a segment has none)
__device__ __forceinline__ void quad_bias(const GemmParams& p, int64_t col, float (&bias)[4]) {
    if (!(p.b0 || p.b1 || p.b2)) return;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int64_t c = col + r < p.N ? col + r : p.N - 1;
        const uint16_t* b = c < p.n0 ? p.b0 : (c < p.n01 ? p.b1 : p.b2);
        if (b) bias[r] = bf2f(b[c < p.n0 ? c : (c < p.n01 ? c - p.n0 : c - p.n01)]);
    }
}

// What the epilogue kEpiQkv loads for a quad of columns at `at`: biases; (cos, sin) of its two pairs in each of the lane's rows
template <int NI>
struct QkvOps {
    float bias[4];
    float4 turn[NI];
};
template <int NI>
__device__ __forceinline__ void qkv_load(const GemmParams& p, const QkvTail& t, int64_t row0, int64_t col, QkvOps<NI>& o) {
    const int hd = 1 << t.hd_log2, at = (int)(col < p.N ? col : p.N - 4);
    o.bias[0] = o.bias[1] = o.bias[2] = o.bias[3] = 0.f;
    quad_bias(p, at, o.bias);
#pragma unroll
    for (int i = 0; i < NI; i++) {   // (no bounds tests: every row's clamped position has them)
        const uint32_t row = (uint32_t)(row0 + 16 * i < p.M ? row0 + 16 * i : p.M - 1);
        o.turn[i] = *reinterpret_cast<const float4*>(t.turns + (int64_t)(row % (uint32_t)t.len) * hd + (at & (hd - 1)));
    }
}
// The epilogue of rows row0 + 16 i, columns col0 + 16 j .. + 3 (whole quads: heads are multiples of 8).  `early`: operands loaded
// ahead, where they are few enough to hold.  A kernel of its own for this (10 us at 2,048 rows, 4 at 113) read the projection back and
// cost a launch.  A layer with this is shorter by: Qwen2-0.5B at 113 rows 2.6 us, Qwen2-7B at 301 rows 5.0, at 2,048 rows 6.3 (there the
// epilogue takes some of it back: with the two tables apart, twice the loads, nothing was left), at 8,192 rows nothing.
template <int NI, int NJ, bool EARLY>
__device__ __forceinline__ void qkv_tail(const GemmParams& p, const QkvTail& t, int64_t row0, int64_t col0, const f32x4 (&acc)[NI][NJ],
                                         const QkvOps<NI> (&early)[EARLY ? NJ : 1]) {
#pragma clang fp contract(off)
    const int hd = 1 << t.hd_log2, turned = t.qd + t.kd;
    int64_t kv[NI];   // where the row's token lies in a run
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const uint32_t row = (uint32_t)(row0 + 16 * i < p.M ? row0 + 16 * i : p.M - 1), seq = row / (uint32_t)t.len;
        const int pos = (int)(row - seq * (uint32_t)t.len);
        kv[i] = t.km.table ? kv_tok<true>(t.km, seq, pos, hd) : kv_tok<false>(t.km, seq, pos, hd);
    }
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int64_t col = col0 + 16 * j;
        const int at = (int)(col < p.N ? col : p.N - 4);
        QkvOps<NI> late;
        if constexpr (!EARLY) qkv_load(p, t, row0, col, late);
        const QkvOps<NI>& o = EARLY ? early[EARLY ? j : 0] : late;
        const int in_kv = at < t.qd ? 0 : at < turned ? at - t.qd : at - turned;
        uint16_t* run = (at < turned ? t.k : t.v) + kv_run_off(t.km, in_kv >> t.hd_log2, hd) + (in_kv & (hd - 1));
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int64_t row = row0 + 16 * i;
            const float4 w = o.turn[i];
            float x[4], y[4];
#pragma unroll
            for (int r = 0; r < 4; r++) x[r] = rbf(acc[i][j][r] + o.bias[r]);
            y[0] = x[0] * w.x - x[1] * w.y;
            y[1] = x[1] * w.x + x[0] * w.y;
            y[2] = x[2] * w.z - x[3] * w.w;
            y[3] = x[3] * w.z + x[2] * w.w;
            uint2 out = make_uint2(pack2(y[0], y[1]), pack2(y[2], y[3]));
            if (at >= turned) out = make_uint2(pack2(x[0], x[1]), pack2(x[2], x[3]));
            if (row < p.M && col < p.N) *reinterpret_cast<uint2*>(at < t.qd ? t.q + row * t.qd + at : run + kv[i]) = out;
        }
    }
}

typedef unsigned int u32x4_g8 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2_g8 __attribute__((ext_vector_type(2)));

// split-K workspace of one launch (gemm8_kernel has the protocol)
struct G8Split {
    int splitk;
    float* slab;       // [tiles][splitk][256 * 256] fp32
    unsigned* cnt;     // tickets, zero at rest; a tile's eight waves' in lines of their own
};
constexpr int G8_TICKET = 16;   // words of a ticket: a line
// (with four ints the arguments of the GEMM kernels: three lines of the segment, and the grid's size behind them in the third)
static_assert(sizeof(GemmParams) + 4 * sizeof(int) + sizeof(G8Split) + 8 + 4 <= 192, "arguments of the GEMM kernels");

// Slabs of 65,536 floats and zeroed tickets of stream `st`, grown on demand; non-zero: they would have to grow during a
// graph capture, or there is no memory (the caller runs unsplit).  What a capture was given stays valid until g8_release.
int g8_workspace(hipStream_t st, int slabs, int tiles, G8Split* out);
// Makes room ahead of the first launch, where a stream is made that will run them.
void g8_reserve(hipStream_t st);
// Gives a stream's split-K memory back: before the engine that owns the stream destroys it, its batches' graphs gone.
void g8_release(hipStream_t st);

// k_gemm_mid.hip: the GEMM of a few dozen to about a thousand rows, and of more where its tiles are the faster (mid::choose; *launched = false: not
// such a shape).  tail: null, or what follows the product.
int gemm_mid(const qie_linear_args* a, const GemmParams& p, const QkvTail* tail, hipStream_t st, bool* launched);
// k_gemm_few.hip: the GEMM of small products (few::choose; *launched = false: not such a shape)
int gemm_few(const qie_linear_args* a, const GemmParams& p, const QkvTail* tail, hipStream_t st, bool* launched);
// One launch of a tile of k_gemm_mid.hip or a form of k_gemm_few.hip, every tile in sk.splitk parts of K whose sums go to sk.slab (kEpiParts).  N a
// multiple of 4, parts below 2^31 bytes.
int gemm_mid_parts(const GemmParams& p, int tile, const G8Split& sk, hipStream_t st);
int gemm_few_parts(const GemmParams& p, int form, const G8Split& sk, hipStream_t st);
// The same for the last columns of a product whose first the 256x256 kernel takes (mid::columns_ahead): always launched.
int gemm_mid_rest(int epi, const GemmParams& p, hipStream_t st);

}  // namespace qie
