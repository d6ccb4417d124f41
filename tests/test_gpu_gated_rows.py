"""Steps of 2 to 16 rows of layered bf16 engines, whose gate and up product has the activation in its epilogue (k_decode_bf16.hip kEpiGated),
against the float64 restatements: every activation; beside the mixer's rows in one product and alone; gate rows that are no whole tiles, mixer
rows that are none; rows of X in LDS and through the ring (width 5,248).  Held to the bf16 engines' tolerance."""
import ctypes as C

import numpy as np
import pytest

import gpu_util as G
import test_gpu_layered as tivazen
import test_gpu_nukizen as nukizen
import test_gpu_sefelorn as sefelorn
import test_gpu_verelorn as verelorn
from nukizen_oracle import att, dense, lru, par
from qwen_inference_engine_amd import _lib
from test_gpu_gemm_mid import bf16, linear

pytestmark = pytest.mark.gpu

MODELS = {
    "relu beside the mixer": (nukizen, [lru(width=30, mlp=dense(24)), att(mlp=dense(1000)), par(mlp=dense(8))], 640),
    "relu, wide": (nukizen, [att(mlp=dense(24)), lru(width=30, mlp=dense(40))], 5248),
    "clamped": (sefelorn, sefelorn.MIXED, 640),
    "gelu": (verelorn, verelorn.MIXED, 640),
    "silu": (tivazen, [tivazen.att(mlp=("dense", 40)), tivazen.att(mlp=("dense", 1000))], 640),
}


@pytest.mark.parametrize("name", MODELS)
def test_few_rows(name):
    mod, layers, width = MODELS[name]
    m = mod.Model(layers, seed=17, dtype="bfloat16", width=width)
    try:
        toks = m.tokens(60)
        want = m.ref(toks)
        got = mod.feed(m, 0, toks, [2, 16, 9, 3, 8, 15, 5, 2])
        d = np.sqrt(((got - want) ** 2).mean(axis=-1)) / np.std(want)
        assert max(np.quantile(d, 0.9), d.max() / 4) < m.tol
        # four slots' rows in one step
        for i in range(1, 4):
            m.batch.step([(i, toks[:20])], [19])
        at = m.batch.step([(i, toks[20:20 + n]) for i, n in ((1, 4), (2, 1), (3, 3))], range(8))
        ref = np.concatenate([want[20:24], want[20:21], want[20:23]])
        d = np.sqrt(((at - ref) ** 2).mean(axis=-1)) / np.std(want)
        assert max(np.quantile(d, 0.9), d.max() / 4) < m.tol
    finally:
        m.close()


class GatedP(C.Structure):   # csrc/k_layered.hpp lay::GatedP
    _fields_ = [("x", C.c_void_p), ("w", C.c_void_p), ("M", C.c_int), ("K", C.c_int), ("plain", C.c_int), ("ff", C.c_int), ("y", C.c_void_p), ("ldy", C.c_int64),
                ("h", C.c_void_p), ("ldh", C.c_int64), ("act", C.c_int), ("limit", C.c_float)]


@pytest.mark.parametrize("act,limit", [(0, 0.0), (1, 0.0), (2, 0.7), (3, 0.0)])
@pytest.mark.parametrize("K,plain,ff,pad", [(640, 0, 30, 3), (640, 36, 1000, 0), (2048, 2052, 2821, 1), (5120, 4, 8, 4), (5248, 0, 40, 0), (5248, 1028, 500, 2)])
def test_as_the_product_and_its_activation(qlib, K, plain, ff, pad, act, limit):
    """lay::GatedP against qie_linear's fp32 product and lay::silu_mul: the same bits, X in LDS (K up to 5,120) and through the ring; nothing behind a
    row's columns."""
    lib = C.CDLL(qlib._name)
    gated, silu = lib._ZN3qie14dec_bf16_gatedERKNS_3lay6GatedPEP12ihipStream_tPb, lib._ZN3qie3lay8silu_mulEPKfPfPtliP12ihipStream_tifll
    silu.argtypes = [C.c_void_p] * 3 + [C.c_int64, C.c_int, C.c_void_p, C.c_int, C.c_float, C.c_int64, C.c_int64]
    rows = plain + 2 * ff
    n_in = (rows + 3) // 4 * 4
    w = bf16((rows, K), 2.0 * K ** -0.5, act + 1)
    dw = G.dev(w)
    for M in (2, 7, 8, 9, 16):
        x = G.dev(bf16((M, K), 1.0, M))
        prod, want, ldh = G.zeros((M, n_in), np.float32), G.zeros_bf16(M, ff), ff + pad
        linear(x, [dw], [], M, K, rows, prod, _lib.QIE_EPI_F32, ldy=n_in)
        G.check(silu(G.p(prod) + plain * 4, None, G.p(want), M, ff, None, act, limit, 0, n_in))
        y, h = G.dev(np.full((M + 1, n_in), 7.0, np.float32)), G.dev(np.full((M + 1, ldh), 0x4040, np.uint16))
        done = C.c_bool(False)
        p = GatedP(G.p(x), G.p(dw), M, K, plain, ff, G.p(y), n_in, G.p(h), ldh, act, limit)
        G.check(gated(C.byref(p), None, C.byref(done)))
        assert done.value, M
        got, gy, prod = h.numpy(), y.numpy(), prod.numpy()
        assert np.array_equal(got[:M, :ff], want.numpy()), M
        assert (got[:M, ff:] == 0x4040).all() and (got[M] == 0x4040).all()
        assert np.array_equal(gy[:M, :plain].view(np.uint32), prod[:, :plain].view(np.uint32))
        assert (gy[:M, plain:] == 7.0).all() and (gy[M] == 7.0).all()
