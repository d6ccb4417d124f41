// k_sum_norm.hip — a product with a residual and the RMSNorm behind it, for prompts: the product's parts of K are added up by the norm's launch.
//
//   x = bf16(x + bf16(A . W^T)), y = RMSNorm(x)     (rmsnorm_reg_kernel's arithmetic and order)
//
// A product of some hundred rows fills the chip only when K is cut.  Meeting in the product's launch, the last workgroup of a tile reads the other
// parts one after the other, 3 us each for 128 x 128 outputs, so products stayed in few parts and small tiles.  The norm's launch is there anyway, has a block for
// every row on all CUs, and reads the row again as soon as it is written: it reads the parts instead (fp32, in part order: the result does not depend on
// anything's arrival).  What bounds it is those bytes: 301 rows of 3,584 in 11 parts, 47 MB, take 8 us (the norm alone 4.4), in one part 4.5.
#include "gemm_impl.hpp"
#include "gemm_plan.hpp"

namespace qie {

// Block per row; thread t has the 8 columns from 8 (t + 256 c) on, as in rmsnorm_reg_kernel
template <int V>
__global__ __launch_bounds__(256) void sum_norm_kernel(const float* __restrict__ sums, int64_t part_at, int parts, uint4* __restrict__ x,
                                                       const uint4* __restrict__ w, uint4* __restrict__ y, int H8, float eps, int numerics) {
    __shared__ float red[4];
    const int tid = threadIdx.x;
    uint4* xr = x + (int64_t)blockIdx.x * H8;
    const float4* sr = reinterpret_cast<const float4*>(sums) + (int64_t)blockIdx.x * H8 * 2;
    part_at /= 4;
    int at[V];
    uint4 xv[V], wv[V];
#pragma unroll
    for (int c = 0; c < V; c++) {
        const int i = tid + 256 * c;
        at[c] = i < H8 ? i : H8 - 1;   // clamped: loads stay unconditional
        xv[c] = xr[at[c]];
        wv[c] = w[at[c]];
    }
    constexpr int FLY = V <= 2 ? 6 : 3;   // parts on their way at a time
    float s[V][8];
    for (int q0 = 0; q0 < parts; q0 += FLY) {
        float4 a[FLY][V], b[FLY][V];
#pragma unroll
        for (int q = 0; q < FLY; q++) {
            const int64_t p = (q0 + q < parts ? q0 + q : parts - 1) * part_at;
#pragma unroll
            for (int c = 0; c < V; c++) {
                a[q][c] = sr[p + at[c] * 2];
                b[q][c] = sr[p + at[c] * 2 + 1];
            }
        }
#pragma unroll
        for (int q = 0; q < FLY; q++) {
            if (q0 + q >= parts) break;   // uniform
#pragma unroll
            for (int c = 0; c < V; c++) {
                const float v[8] = {a[q][c].x, a[q][c].y, a[q][c].z, a[q][c].w, b[q][c].x, b[q][c].y, b[q][c].z, b[q][c].w};
#pragma unroll
                for (int j = 0; j < 8; j++) s[c][j] = q0 + q == 0 ? v[j] : s[c][j] + v[j];
            }
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < V; c++) {
        uint32_t e[4] = {xv[c].x, xv[c].y, xv[c].z, xv[c].w};
#pragma unroll
        for (int j = 0; j < 4; j++) e[j] = pack2(bf_lo(e[j]) + rbf(s[c][2 * j]), bf_hi(e[j]) + rbf(s[c][2 * j + 1]));
        xv[c] = make_uint4(e[0], e[1], e[2], e[3]);
        if (tid + 256 * c >= H8) continue;
        xr[at[c]] = xv[c];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float l = bf_lo(e[j]), h = bf_hi(e[j]);
            ss += l * l + h * h;
        }
    }
    ss = wave_sum(ss);
    if ((tid & 63) == 0) red[tid >> 6] = ss;
    __syncthreads();
    ss = red[0] + red[1] + red[2] + red[3];
    const float rms = sqrtf((ss / (float)(8 * (int64_t)H8)) + eps), inv = 1.0f / rms;
    uint4* yr = y + (int64_t)blockIdx.x * H8;
#pragma unroll
    for (int c = 0; c < V; c++) {
#pragma clang fp contract(off)
        if (tid + 256 * c >= H8) continue;
        const uint32_t e[4] = {xv[c].x, xv[c].y, xv[c].z, xv[c].w}, n[4] = {wv[c].x, wv[c].y, wv[c].z, wv[c].w};
        uint32_t o[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (numerics == QIE_NUMERICS_HF) o[j] = pack2(bf_lo(n[j]) * rbf(bf_lo(e[j]) * inv), bf_hi(n[j]) * rbf(bf_hi(e[j]) * inv));
            else o[j] = pack2((bf_lo(e[j]) / rms) * bf_lo(n[j]), (bf_hi(e[j]) / rms) * bf_hi(n[j]));
        }
        yr[at[c]] = make_uint4(o[0], o[1], o[2], o[3]);
    }
}

// The product `a` (checked; RESIDUAL, rows of N in a->y without gaps, one weight segment) and y = the norm of its rows
int gemm_add_norm(const qie_linear_args* a, const void* norm_w, float eps, int numerics, void* y, hipStream_t st) {
    const int64_t vectors = a->N % 8 == 0 ? (a->N / 8 + 255) / 256 : 0;
    const bool fits = a->M > 16 && !(a->flags & (QIE_LINEAR_FP8 | QIE_LINEAR_FP8_T16 | QIE_LINEAR_ACT_FP8)) && !a->norm_w && a->seg_rows[0] == a->N && a->ldy == a->N &&
                      vectors >= 1 && vectors <= 4 && mid::strides_fit(a->ldx, a->ldy) && ((uintptr_t)a->y | (uintptr_t)norm_w | (uintptr_t)y) % 16 == 0 && a->y != y;
    const apart::Plan pl = fits && dev_env("QIE_APART", 1) ? apart::choose(a->M, a->N, a->K, device_cu_count()) : apart::Plan{-1, -1, 1, 0.f};
    G8Split sk{pl.parts, nullptr, nullptr};
    if ((pl.form < 0 && pl.tile < 0) || g8_workspace(st, cdiv(pl.parts * a->M * a->N, 65536), 1, &sk) != 0) {
        QIE_TRY(qie_linear(a, st));
        return qie_rmsnorm(a->y, norm_w, y, a->M, a->N, eps, numerics, st);
    }
    sk.splitk = pl.parts;
    GemmParams p{};
    p.A = (const uint16_t*)a->x;
    p.lda = a->ldx;
    p.w0 = p.w1 = p.w2 = (const uint16_t*)a->w[0];
    p.n0 = p.n01 = a->N;
    p.M = a->M;
    p.K = a->K;
    p.N = a->N;
    QIE_TRY(pl.form >= 0 ? gemm_few_parts(p, pl.form, sk, st) : gemm_mid_parts(p, pl.tile, sk, st));
    auto fn = vectors <= 1 ? sum_norm_kernel<1> : vectors <= 2 ? sum_norm_kernel<2> : vectors <= 3 ? sum_norm_kernel<3> : sum_norm_kernel<4>;
    hipLaunchKernelGGL(fn, dim3((unsigned)a->M), dim3(256), 0, st, sk.slab, a->M * a->N, pl.parts, (uint4*)a->y, (const uint4*)norm_w, (uint4*)y, (int)(a->N / 8), eps,
                       numerics);
    QIE_LAUNCH_CHECK();
    return 0;
}

}  // namespace qie
