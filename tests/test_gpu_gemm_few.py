"""The GEMM of small products (k_gemm_few.hip) through qie_linear, against fp32 products: every form at the edges of its tiles, K of fewer chunks than
waves, of one more and of many, each epilogue, odd columns and row strides, segments that its tiles would cross."""
import os
import subprocess

import numpy as np
import pytest

import gpu_util as G
from qwen_inference_engine_amd import _lib
from test_gpu_gemm_mid import bf16, linear, products

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen_inference_engine_amd", "csrc")
DRIVER = r"""
#include "gemm_plan.hpp"
#include <cstdio>
int main() {
    long M, cols, K, gated, ragged;
    while (std::scanf("%ld %ld %ld %ld %ld", &M, &cols, &K, &gated, &ragged) == 5)
        std::printf("%d\n", qie::few::choose(M, cols, K, 256, gated != 0, ragged != 0).form);
}
"""
# rows, columns, K, form: tiles of 32 x 16, 32 x 32, 32 x 64, 64 x 32, 64 x 64
SHAPES = [(17, 1152, 896, 0), (33, 1000, 2048, 0), (64, 16, 1024, 0), (113, 1152, 896, 1), (32, 5632, 1024, 1), (129, 1153, 320, 1), (65, 4608, 3584, 2),
          (400, 1153, 640, 2), (129, 2000, 960, 3), (256, 2048, 1536, 3), (510, 2047, 2048, 4)]


def forms(tmp_path, cases):
    (tmp_path / "drive.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "drive.cpp"), "-o", str(tmp_path / "drive")], check=True)
    out = subprocess.run([str(tmp_path / "drive")], input="\n".join("%d %d %d %d %d" % c for c in cases), text=True, capture_output=True, check=True).stdout
    return [int(v) for v in out.split()]


def test_shapes_take_every_form(tmp_path):
    got = forms(tmp_path, [(*s[:3], 0, 0) for s in SHAPES])
    assert got == [s[3] for s in SHAPES] and set(got) == set(range(5))
    # gate and up: 32 rows at most; never K off the grid of 64, segments that tiles would cross, or rows beyond the fit
    assert forms(tmp_path, [(32, 9728, 896, 1, 0), (24, 37888, 3584, 1, 0), (33, 9728, 896, 1, 0)]) == [2, 1, -1]
    assert forms(tmp_path, [(113, 1152, 928, 0, 0), (113, 1152, 896, 0, 1), (513, 1152, 896, 0, 0), (301, 37888, 3584, 1, 0)]) == [-1] * 4


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [s[:3] for s in SHAPES])
def test_products(qlib, M, N, K):
    x, w = bf16((M, K), 1.0, 1), bf16((N, K), K ** -0.5, 2)
    y = G.zeros((M, N), np.float32)
    linear(G.dev(x), [G.dev(w)], [], M, K, N, y, _lib.QIE_EPI_F32)
    want, scale = products(x, w)
    # two fp32 sums of K products in different orders: each within 2^-24 sqrt(K)-ish of the exact one, 1e-5 of the absolute sum holds both
    assert (np.abs(y.numpy() - want) <= 1e-5 * scale).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,K", [(17, 64), (32, 320), (31, 896), (24, 2048)])
@pytest.mark.parametrize("n", [200, 197, 8201])
def test_gated(qlib, M, K, n):
    """Gate and up of up to 32 rows: one round of 32 x 64 tiles, and more of 32 x 32."""
    x, wg, wu = bf16((M, K), 1.0, 3), bf16((n, K), 1.5 * K ** -0.5, 4), bf16((n, K), K ** -0.5, 5)
    y = G.zeros_bf16(M, n)
    linear(G.dev(x), [G.dev(wg), G.dev(wu)], [], M, K, n, y, _lib.QIE_EPI_SWIGLU)
    (g, gs), (u, us) = products(x, wg), products(x, wu)
    want = u / (1.0 + np.exp(-g)) * g
    # |silu'| <= 1.1; three bf16 roundings (gate, silu, product) and one of the up sum
    tol = 2.0 ** -7 * (np.abs(want) + 1.1 * np.abs(u) * np.abs(g)) + 1e-5 * (1.1 * np.abs(u) * gs + np.abs(g) * us)
    assert (np.abs(G.bf(G.host_bf16(y)) - want) <= tol).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,rows", [(33, (128, 64, 64)), (113, (64, 64, 40)), (113, (64, 64, 41)), (113, (132, 72, 40))])
def test_segments(qlib, oracle, M, rows):
    """Biases of three segments: whole tiles of each, a last one that is not, and (the others' kernel) tiles across them."""
    K = 896
    x, ws, bs = bf16((M, K), 1.0, 3), [bf16((r, K), K ** -0.5, 4 + i) for i, r in enumerate(rows)], [bf16((r,), 0.5, 7 + i) for i, r in enumerate(rows)]
    N = sum(rows)
    y = G.zeros_bf16(M, N)
    linear(G.dev(x), [G.dev(w) for w in ws], [G.dev(b) for b in bs], M, K, N, y, _lib.QIE_EPI_STORE)
    want, scale = products(x, np.concatenate(ws))
    G.assert_sum_close(G.host_bf16(y), oracle.f32_to_bf16((want + G.bf(np.concatenate(bs))).astype(np.float32)), scale, what="segments")


@pytest.mark.gpu
@pytest.mark.parametrize("N,ld", [(264, 264), (261, 263)])
def test_residual(qlib, oracle, N, ld):
    """Rows of x and y at strides of their own; nothing behind the row's columns; repeated calls give the same bits."""
    M, K, ldx = 50, 960, 968
    x, w, res = bf16((M, ldx), 1.0, 3), bf16((N, K), K ** -0.5, 4), bf16((M, ld), 1.0, 5)
    got = []
    for _ in range(2):
        y = G.dev(res)
        linear(G.dev(x), [G.dev(w)], [], M, K, N, y, _lib.QIE_EPI_RESIDUAL, ldx=ldx, ldy=ld)
        got.append(G.host_bf16(y))
    acc, scale = products(x[:, :K], w)
    want = G.bf(res)[:, :N] + G.bf(oracle.f32_to_bf16(acc))
    tol = 2.0 ** -7 * (np.abs(acc) + np.abs(want)) + 1e-5 * scale   # bf16(res + bf16(acc)): an ulp of either rounding
    assert (np.abs(G.bf(got[0])[:, :N] - want) <= tol).all()
    assert np.array_equal(got[0][:, N:], res[:, N:]) and np.array_equal(got[0], got[1])
