"""One-row projections with a whole weight row in a wave's registers (k_gemv_row.hip) through qie_linear, against fp32 products:
K at the edges of the register forms, rows from one to 32 a CU, segments, every epilogue it takes, the fused norm in both numerics."""
import ctypes as C

import numpy as np
import pytest

import gpu_util as G
from qwen_inference_engine_amd import _lib
from test_gpu_gemm_mid import bf16, linear, products

pytestmark = pytest.mark.gpu

KS = [8, 896, 1024, 1032, 2048, 2056, 3584, 3592, 4864, 5120]


@pytest.mark.parametrize("K", KS)
@pytest.mark.parametrize("N", [1, 5, 1153, 4700, 8191])   # 8,192 rows are 32 a CU on 256; the grid's last block ragged
def test_products(qlib, K, N):
    x, w = bf16((1, K), 1.0, 1), bf16((N, K), K ** -0.5, 2)
    dx, dw, y = G.dev(x), G.dev(w), G.zeros((1, N), np.float32)
    linear(dx, [dw], [], 1, K, N, y, _lib.QIE_EPI_F32)
    want, scale = products(x, w)
    assert (np.abs(y.numpy() - want) <= 1e-5 * scale).all()   # two orders of one fp32 sum


@pytest.mark.parametrize("K", KS)
def test_epilogues(qlib, oracle, K):
    x = bf16((1, K), 1.0, 3)
    n = (133, 70, 42)
    ws, bs = [bf16((r, K), K ** -0.5, 4 + i) for i, r in enumerate(n)], [bf16((r,), 0.5, 7 + i) for i, r in enumerate(n)]
    y = G.zeros_bf16(1, sum(n))
    linear(G.dev(x), [G.dev(w) for w in ws], [G.dev(b) for b in bs], 1, K, sum(n), y, _lib.QIE_EPI_STORE)
    want, scale = products(x, np.concatenate(ws))
    G.assert_sum_close(G.host_bf16(y), oracle.f32_to_bf16((want + G.bf(np.concatenate(bs))).astype(np.float32)), scale, what="store")
    w, res = bf16((261, K), K ** -0.5, 4), bf16((1, 264), 1.0, 5)
    y = G.dev(res)
    linear(G.dev(x), [G.dev(w)], [], 1, K, 261, y, _lib.QIE_EPI_RESIDUAL, ldy=264)
    got = G.host_bf16(y)
    acc, scale = products(x, w)
    want = G.bf(res)[:, :261] + G.bf(oracle.f32_to_bf16(acc))
    tol = 2.0 ** -7 * (np.abs(acc) + np.abs(want)) + 1e-5 * scale   # an ulp of either rounding
    assert (np.abs(G.bf(got)[:, :261] - want) <= tol).all() and np.array_equal(got[:, 261:], res[:, 261:])


@pytest.mark.parametrize("K", KS)
@pytest.mark.parametrize("N", [70, 4700, 8191])
@pytest.mark.parametrize("num", ["ref", "hf"])
def test_norm(qlib, oracle, K, N, num):
    eps = 1e-4 if num == "ref" else 1e-6
    x, nw, w = bf16((1, K), 1.0, 11), bf16((K,), 0.2, 12), bf16((N, K), K ** -0.5, 13)
    nw = oracle.f32_to_bf16(1.0 + G.bf(nw))
    x[0, :K // 4] = 0
    xn = oracle.rmsnorm(x, nw, eps, num)
    dx, dw, dn, y = G.dev(x), G.dev(w), G.dev(nw), G.zeros_bf16(1, N)
    a = _lib.LinearArgsC()
    a.x, a.ldx, a.w[0], a.seg_rows[0], a.M, a.K, a.N = G.p(dx), K, G.p(dw), N, 1, K, N
    a.y, a.ldy, a.epilogue, a.numerics, a.norm_w, a.norm_eps = G.p(y), N, _lib.QIE_EPI_STORE, 0 if num == "ref" else 1, G.p(dn), eps
    G.check(qlib.qie_linear(C.byref(a), None), "qie_linear")
    want, scale = products(xn, w)
    # a normed element may round to the neighbouring bf16 (another order of the row's sum of squares): 2^-8 of its share, seldom
    assert (np.abs(G.bf(G.host_bf16(y)) - want) <= 2.0 ** -7 * np.abs(want) + 1e-3 * scale).all()
