// gemm_impl.hpp — what the prefill GEMMs share (k_gemm.hip, k_gemm_mid.hip): operands, LDS-DMA, the split-K workspace.
#pragma once

#include "qie_common.hpp"
#include "../../include/qie/qie_ops.h"
#include "split_pool.hpp"

namespace qie {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

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
__device__ __forceinline__ void add_quad(uint16_t* dst, uint2 x, f32x4 v, bool vec, int64_t left) {
    const float o[4] = {bf_lo(x.x) + rbf(v[0]), bf_hi(x.x) + rbf(v[1]), bf_lo(x.y) + rbf(v[2]), bf_hi(x.y) + rbf(v[3])};
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

typedef unsigned int u32x4_g8 __attribute__((ext_vector_type(4)));

// split-K workspace of one launch (gemm8_kernel has the protocol)
struct G8Split {
    int splitk;
    float* slab;       // [tiles][splitk][256 * 256] fp32
    unsigned* cnt;     // [tiles], zero at rest
};

// Slabs of 65,536 floats and zeroed tickets of stream `st`, grown on demand; non-zero: they would have to grow during a
// graph capture, or there is no memory (the caller runs unsplit).  What a capture was given stays valid until g8_release.
int g8_workspace(hipStream_t st, int slabs, int tiles, G8Split* out);
// Makes room ahead of the first launch, where a stream is made that will run them.
void g8_reserve(hipStream_t st);
// Gives a stream's split-K memory back: before the engine that owns the stream destroys it, its batches' graphs gone.
void g8_release(hipStream_t st);

// k_gemm_mid.hip: the GEMM of a few dozen to about a thousand rows.  other_us: the expected time of the caller's kernel for
// this shape; *launched = false: not a shape for this one, or the other is expected to be faster.
int gemm_mid(const qie_linear_args* a, const GemmParams& q, float other_us, hipStream_t st, bool* launched);

}  // namespace qie
