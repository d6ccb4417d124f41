"""The prefill GEMMs over so many row tiles that their workgroups take them in bands, against fp32 products: a last band and a last
tile of fewer rows, the last columns' tile partly empty."""
import ctypes as C

import numpy as np
import pytest

import gpu_util as G
from qwen_inference_engine_amd import _lib
from test_gpu_gemm_mid import bf16, products

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flags", [0, _lib.QIE_LINEAR_TILE256])
@pytest.mark.parametrize("M,N,K", [(4400, 1100, 256), (6151, 300, 320)])
def test_products(qlib, M, N, K, flags):
    x, w = bf16((M, K), 1.0, 1), bf16((N, K), K ** -0.5, 2)
    y = G.zeros((M, N), np.float32)
    a = _lib.LinearArgsC()
    dx, dw = G.dev(x), G.dev(w)
    a.x, a.ldx, a.w[0], a.seg_rows[0] = G.p(dx), K, G.p(dw), N
    a.M, a.K, a.N, a.y, a.ldy, a.epilogue, a.flags = M, K, N, G.p(y), N, _lib.QIE_EPI_F32, flags
    G.check(_lib.load().qie_linear(C.byref(a), None), "qie_linear")
    want, scale = products(x, w)
    # two fp32 sums of K products in different orders
    assert (np.abs(y.numpy() - want) <= 1e-5 * scale).all()


@pytest.mark.parametrize("M,N,K", [(300, 261, 256), (511, 520, 320)])   # scalar stores and a row stride of its own; vector stores
@pytest.mark.parametrize("epi", ["store", "residual", "swiglu"])
def test_epilogues_of_256_tiles(qlib, oracle, M, N, K, epi):
    ld = N + N % 2 * 2
    x, res = bf16((M, K), 1.0, 3), bf16((M, ld), 1.0, 5)
    ws = [bf16((N, K), (1.5 - 0.5 * i) * K ** -0.5, 4 + i) for i in range(2 if epi == "swiglu" else 1)]
    y, dx, dw, db = G.dev(res), G.dev(x), [G.dev(w) for w in ws], G.dev(bf16((N,), 0.5, 7))
    a = _lib.LinearArgsC()
    a.x, a.ldx, a.M, a.K, a.N, a.y, a.ldy, a.flags = G.p(dx), K, M, K, N, G.p(y), ld, _lib.QIE_LINEAR_TILE256
    for i, w in enumerate(dw):
        a.w[i], a.seg_rows[i] = G.p(w), N
    a.epilogue = {"store": _lib.QIE_EPI_STORE, "residual": _lib.QIE_EPI_RESIDUAL, "swiglu": _lib.QIE_EPI_SWIGLU}[epi]
    if epi == "store":
        a.bias[0] = G.p(db)
    G.check(_lib.load().qie_linear(C.byref(a), None), "qie_linear")
    got = G.host_bf16(y)
    assert np.array_equal(got[:, N:], res[:, N:])   # nothing behind the row's columns
    got, (v, scale) = G.bf(got)[:, :N], products(x, ws[0])
    if epi == "swiglu":
        u, us = products(x, ws[1])
        want = u / (1.0 + np.exp(-v)) * v
        # |silu'| <= 1.1; three bf16 roundings (gate, silu, product) and one of the up sum
        tol = 2.0 ** -7 * (np.abs(want) + 1.1 * np.abs(u) * np.abs(v)) + 1e-5 * (1.1 * np.abs(u) * scale + np.abs(v) * us)
    else:
        want = v + G.bf(bf16((N,), 0.5, 7)) if epi == "store" else G.bf(res)[:, :N] + G.bf(oracle.f32_to_bf16(v))
        tol = 2.0 ** -7 * (np.abs(v) + np.abs(want)) + 1e-5 * scale   # an ulp of either rounding
    assert (np.abs(got - want) <= tol).all()
