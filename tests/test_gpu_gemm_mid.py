"""The GEMM of a few dozen to about a thousand rows (k_gemm_mid.hip) through qie_linear, against fp32 products: shapes whose
plan takes every tile, whole, split and mixed, at ragged rows and columns; odd columns and row strides (scalar stores); every
epilogue."""
import ctypes as C

import numpy as np
import pytest

import gpu_util as G
from qwen_inference_engine_amd import _lib

pytestmark = pytest.mark.gpu

POOL = np.random.default_rng(5).standard_normal((1 << 20) + 7).astype(np.float32)


def bf16(shape, scale, seed):
    """bf16 words of a shape, drawn from one pool of normals."""
    n = int(np.prod(shape))
    v = np.resize(np.roll(POOL, 7919 * seed), n).reshape(shape) * np.float32(scale)
    u = v.view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def products(x, w):
    a, b = G.bf(x).astype(np.float32), G.bf(w).astype(np.float32)
    return a @ b.T, np.abs(a) @ np.abs(b).T


def linear(x, ws, biases, M, K, N, y, epi, ldx=None, ldy=None):
    a = _lib.LinearArgsC()
    a.x, a.ldx = G.p(x), ldx or K
    for i, w in enumerate(ws):
        a.w[i], a.seg_rows[i] = G.p(w), w.shape[0]
    for i, b in enumerate(biases):
        a.bias[i] = G.p(b)
    a.M, a.K, a.N, a.y, a.ldy, a.epilogue = M, K, N, G.p(y), ldy or N, epi
    G.check(_lib.load().qie_linear(C.byref(a), None), "qie_linear")


# rows, columns, K; the tile that the plan gives them on 256 CUs, and whether tiles run whole, are all split over K, or both
# (tests/test_gemm_plan.py holds the plan to this, and every tile to all three)
PLANS = [(17, 72, 64, 0, "whole"), (33, 72, 2048, 0, "split"), (17, 40000, 128, 0, "mixed"), (17, 16500, 64, 1, "whole"),
         (64, 8200, 4096, 1, "split"), (65, 40000, 128, 1, "mixed"), (65, 8200, 1024, 2, "whole"), (129, 4000, 4096, 2, "split"),
         (65, 33000, 2048, 2, "mixed"), (127, 16500, 64, 3, "whole"), (128, 8200, 4096, 3, "split"), (193, 40000, 2048, 3, "mixed"),
         (500, 8200, 128, 4, "whole"), (129, 33000, 1024, 1, "whole"), (640, 8200, 448, 5, "whole"), (193, 70000, 512, 1, "whole"),
         (640, 4000, 4096, 6, "split"), (257, 40000, 1024, 1, "mixed"), (257, 16500, 1024, 7, "whole"), (320, 33000, 2048, 1, "whole"),
         (321, 130, 192, 1, "whole"), (140, 38660, 2624, 4, "mixed"), (131, 11014, 3712, 4, "split"), (200, 45648, 1792, 5, "mixed"),
         (210, 9278, 6464, 5, "split"), (273, 38147, 1792, 6, "mixed"), (259, 12692, 64, 6, "whole"), (1064, 11882, 1728, 7, "mixed"),
         (257, 8338, 11264, 7, "split")]
SHAPES = [p[:3] for p in PLANS]
# Other tiles, k_gemm_few.hip or two launches are the better choice for half of those; with these qie_linear comes to every tile in every way that is left
MORE = [(129, 44169, 128), (72, 42624, 2048), (70, 16787, 320), (131, 42200, 2880), (130, 20894, 64), (193, 20859, 448), (261, 47014, 1536), (838, 28106, 64), (33, 72, 12416)]
GROWS = (130, 22370, 17472)   # partial tiles of more than the 64 MB that a stream has from the start


@pytest.mark.parametrize("M,N,K", SHAPES + MORE)
def test_products(qlib, M, N, K):
    x, w = bf16((M, K), 1.0, 1), bf16((N, K), K ** -0.5, 2)
    y = G.zeros((M, N), np.float32)
    linear(G.dev(x), [G.dev(w)], [], M, K, N, y, _lib.QIE_EPI_F32)
    want, scale = products(x, w)
    # two fp32 sums of K products in different orders: each within 2^-24 sqrt(K)-ish of the exact one, 1e-5 of the absolute sum holds both
    assert (np.abs(y.numpy() - want) <= 1e-5 * scale).all()


@pytest.mark.parametrize("M,K", [(17, 64), (64, 896), (113, 4864), (301, 128), (700, 320)])
@pytest.mark.parametrize("epi", ["store", "store odd", "residual", "residual odd", "swiglu", "swiglu odd"])
def test_epilogues(qlib, oracle, M, K, epi):
    odd = epi.endswith("odd")
    x = bf16((M, K), 1.0, 3)
    if epi.startswith("store"):
        n = (133, 70, 42) if odd else (132, 72, 40)   # the bias changes inside a vector of four columns
        ws, bs = [bf16((r, K), K ** -0.5, 4 + i) for i, r in enumerate(n)], [bf16((r,), 0.5, 7 + i) for i, r in enumerate(n)]
        N = sum(n)
        y = G.zeros_bf16(M, N)
        linear(G.dev(x), [G.dev(w) for w in ws], [G.dev(b) for b in bs], M, K, N, y, _lib.QIE_EPI_STORE)
        want, scale = products(x, np.concatenate(ws))
        want = want + G.bf(np.concatenate(bs))
        G.assert_sum_close(G.host_bf16(y), oracle.f32_to_bf16(want.astype(np.float32)), scale, what=epi)
    elif epi.startswith("residual"):
        N, ld = (261, 263) if odd else (264, 264)
        w, res = bf16((N, K), K ** -0.5, 4), bf16((M, ld), 1.0, 5)
        y = G.dev(res)
        linear(G.dev(x), [G.dev(w)], [], M, K, N, y, _lib.QIE_EPI_RESIDUAL, ldy=ld)
        got = G.host_bf16(y)
        acc, scale = products(x, w)
        want = G.bf(res)[:, :N] + G.bf(oracle.f32_to_bf16(acc))
        # bf16(res + bf16(acc)): an ulp of either rounding
        tol = 2.0 ** -7 * (np.abs(acc) + np.abs(want)) + 1e-5 * scale
        assert (np.abs(G.bf(got)[:, :N] - want) <= tol).all()
        assert np.array_equal(got[:, N:], res[:, N:])   # nothing behind the row's columns
    else:
        N = 197 if odd else 200
        wg, wu = bf16((N, K), 1.5 * K ** -0.5, 4), bf16((N, K), K ** -0.5, 5)
        y = G.zeros_bf16(M, N)
        linear(G.dev(x), [G.dev(wg), G.dev(wu)], [], M, K, N, y, _lib.QIE_EPI_SWIGLU)
        (g, gs), (u, us) = products(x, wg), products(x, wu)
        want = u / (1.0 + np.exp(-g)) * g
        # |silu'| <= 1.1; three bf16 roundings (gate, silu, product) and one of the up sum
        tol = 2.0 ** -7 * (np.abs(want) + 1.1 * np.abs(u) * np.abs(g)) + 1e-5 * (1.1 * np.abs(u) * gs + np.abs(g) * us)
        assert (np.abs(G.bf(G.host_bf16(y)) - want) <= tol).all()


def test_row_stride(qlib):
    """Rows of x at a stride of their own; repeated calls give the same bits (split parts in part order)."""
    M, K, N, ldx = 113, 896, 264, 904
    x, w = bf16((M, ldx), 1.0, 6), bf16((N, K), K ** -0.5, 7)
    buf, dw, out = G.dev(x), G.dev(w), []
    for _ in range(3):
        y = G.zeros((M, N), np.float32)
        linear(buf, [dw], [], M, K, N, y, _lib.QIE_EPI_F32, ldx=ldx)
        out.append(y.numpy())
    want, scale = products(x[:, :K], w)
    assert (np.abs(out[0] - want) <= 1e-5 * scale).all()
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])


def test_split_is_deterministic(qlib):
    M, K, N = 301, 4096, 520
    x, w = G.dev(bf16((M, K), 1.0, 8)), G.dev(bf16((N, K), K ** -0.5, 9))
    out = []
    for _ in range(4):
        y = G.zeros((M, N), np.float32)
        linear(x, [w], [], M, K, N, y, _lib.QIE_EPI_F32)
        out.append(y.numpy())
    assert all(np.array_equal(out[0], o) for o in out[1:])


@pytest.mark.parametrize("M,N,K", [(301, 1152, 896), (345, 45029, 768)])
def test_rows_far_apart(qlib, M, N, K):
    """Rows of x whose offsets inside a tile pass 32 bits (4.3 GB of 301 rows), of a product that k_gemm_mid.hip takes whole and of one that it takes
    the last columns of: others do."""
    ld = 7200000
    x, w = bf16((M, K), 1.0, 1), bf16((N, K), K ** -0.5, 2)
    far = G.DBuf((M - 1) * ld + K, np.uint16)
    for m in range(M):
        G.check(qlib.qie_memcpy_h2d(far.ptr + m * ld * 2, x[m].ctypes.data, K * 2))
    y = G.zeros((M, N), np.float32)
    linear(far, [G.dev(w)], [], M, K, N, y, _lib.QIE_EPI_F32, ldx=ld)
    want, scale = products(x, w)
    assert (np.abs(y.numpy() - want) <= 1e-5 * scale).all()
