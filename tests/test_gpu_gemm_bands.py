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
