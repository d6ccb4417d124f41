"""Products of few 256x256 tiles whose K is cut into 2, 3 and 4 parts (k_gemm.hip sum_parts): every epilogue, ragged rows and columns, against
fp32 products, and the same bits whichever part came last."""
import numpy as np
import pytest

import gpu_util as G
from gemm_route import routes
from qwen_inference_engine_amd import _lib
from test_gpu_gemm_mid import bf16, linear, products

# rows, weight rows, K, parts
SHAPES = [(599, 8376, 9280, 2), (782, 4636, 12416, 3), (385, 5660, 21952, 4)]


def test_the_shapes_are_cut():
    assert [(r["tile"], r["parts"], r["ahead"]) for r in routes([s[:3] for s in SHAPES])] == [(-1, s[3], 0) for s in SHAPES]


@pytest.mark.gpu
@pytest.mark.parametrize("M,rows,K,parts", SHAPES)
def test_parts(qlib, oracle, M, rows, K, parts):
    x, w, b = bf16((M, K), 1.0, 31), bf16((rows, K), K ** -0.5, 32), bf16((rows,), 0.5, 33)
    dx, dw, db = G.dev(x), G.dev(w), G.dev(b)
    acc, scale = products(x, w)
    ld, y0 = rows + 3, bf16((M + 1, rows + 3), 1.0, 34)
    first = None
    for _ in range(4):
        y = G.zeros((M, rows), np.float32)
        linear(dx, [dw], [], M, K, rows, y, _lib.QIE_EPI_F32)
        got = y.numpy()
        first = got if first is None else first
        assert np.array_equal(got.view(np.uint32), first.view(np.uint32))
    assert (np.abs(first - acc) <= 1e-5 * scale).all()   # two fp32 sums of K products in different orders
    y = G.dev(y0)
    linear(dx, [dw], [db], M, K, rows, y, _lib.QIE_EPI_STORE, ldy=ld)
    got, want = G.host_bf16(y), acc + G.bf(b)
    assert (np.abs(G.bf(got)[:M, :rows] - want) <= 2.0 ** -8 * np.abs(want) + 1e-5 * scale).all()
    assert np.array_equal(got[:M, rows:], y0[:M, rows:]) and np.array_equal(got[M], y0[M])
    y = G.dev(y0)
    linear(dx, [dw], [], M, K, rows, y, _lib.QIE_EPI_RESIDUAL, ldy=ld)
    got, want = G.host_bf16(y), G.bf(y0)[:M, :rows] + G.bf(oracle.f32_to_bf16(acc))
    # bf16(res + bf16(acc)): an ulp of either rounding
    assert (np.abs(G.bf(got)[:M, :rows] - want) <= 2.0 ** -7 * (np.abs(acc) + np.abs(want)) + 1e-5 * scale).all()
    assert np.array_equal(got[:M, rows:], y0[:M, rows:]) and np.array_equal(got[M], y0[M])
    N = rows // 2   # the same rows as gate and up
    y = G.dev(y0)
    linear(dx, [G.dev(w[:N]), G.dev(w[N:])], [], M, K, N, y, _lib.QIE_EPI_SWIGLU, ldy=ld)
    (g, u), (gs, us) = (acc[:, :N], acc[:, N:]), (scale[:, :N], scale[:, N:])
    got, want = G.host_bf16(y), u / (1.0 + np.exp(-g)) * g
    # |silu'| <= 1.1; three bf16 roundings (gate, silu, product) and one of the up sum
    tol = 2.0 ** -7 * (np.abs(want) + 1.1 * np.abs(u) * np.abs(g)) + 1e-5 * (1.1 * np.abs(u) * gs + np.abs(g) * us)
    assert (np.abs(G.bf(got)[:M, :N] - want) <= tol).all()
    assert np.array_equal(got[:M, N:], y0[:M, N:]) and np.array_equal(got[M], y0[M])
