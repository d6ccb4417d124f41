"""The batched decode projections on bf16 weights (k_decode_bf16.hip) through qie_linear, 2 to 16 rows, against fp32 products:
X in LDS and through the ring, fewer and more tiles than CUs, ragged columns, every epilogue, the fused norm in both numerics,
arg-max keys; K off the 128 grid and too many normed rows stay with the kernels that took them."""
import ctypes as C

import numpy as np
import pytest

import gpu_util as G
from qwen_inference_engine_amd import _lib
from test_gpu_gemm_mid import bf16, linear, products

pytestmark = pytest.mark.gpu



# K / 128 chunks over 8 waves: under one each, one, uneven, X too large for LDS; N: one tile, ragged, more tiles than CUs
@pytest.mark.parametrize("M,K,N", [(2, 512, 16), (2, 896, 72), (3, 1024, 4100), (4, 3584, 130), (5, 4864, 40), (7, 5120, 264), (8, 3584, 9000),
                                   (8, 5120, 48), (8, 17408, 40), (9, 2048, 4200), (13, 5120, 50), (16, 2048, 33), (16, 4864, 264),
                                   (2, 960, 40), (16, 18944, 24)])
def test_products(qlib, M, K, N):
    x, w = bf16((M, K), 1.0, 1), bf16((N, K), K ** -0.5, 2)
    dx, dw, out = G.dev(x), G.dev(w), []
    for _ in range(2):
        y = G.zeros((M, N), np.float32)
        linear(dx, [dw], [], M, K, N, y, _lib.QIE_EPI_F32)
        out.append(y.numpy())
    want, scale = products(x, w)
    assert (np.abs(out[0] - want) <= 1e-5 * scale).all()   # two orders of one fp32 sum
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("M,K", [(2, 896), (4, 3584), (8, 1024), (16, 2048), (6, 17408)])
@pytest.mark.parametrize("epi", ["store", "store odd", "residual", "residual odd", "swiglu", "swiglu odd"])
def test_epilogues(qlib, oracle, M, K, epi):
    odd = epi.endswith("odd")
    x = bf16((M, K), 1.0, 3)
    if epi.startswith("store"):
        n = (133, 70, 42) if odd else (132, 72, 40)
        ws, bs = [bf16((r, K), K ** -0.5, 4 + i) for i, r in enumerate(n)], [bf16((r,), 0.5, 7 + i) for i, r in enumerate(n)]
        N = sum(n)
        y = G.zeros_bf16(M, N)
        linear(G.dev(x), [G.dev(w) for w in ws], [G.dev(b) for b in bs], M, K, N, y, _lib.QIE_EPI_STORE)
        want, scale = products(x, np.concatenate(ws))
        G.assert_sum_close(G.host_bf16(y), oracle.f32_to_bf16((want + G.bf(np.concatenate(bs))).astype(np.float32)), scale, what=epi)
    elif epi.startswith("residual"):
        N, ld = (261, 263) if odd else (264, 264)
        w, res = bf16((N, K), K ** -0.5, 4), bf16((M, ld), 1.0, 5)
        y = G.dev(res)
        linear(G.dev(x), [G.dev(w)], [], M, K, N, y, _lib.QIE_EPI_RESIDUAL, ldy=ld)
        got = G.host_bf16(y)
        acc, scale = products(x, w)
        want = G.bf(res)[:, :N] + G.bf(oracle.f32_to_bf16(acc))
        tol = 2.0 ** -7 * (np.abs(acc) + np.abs(want)) + 1e-5 * scale   # an ulp of either rounding
        assert (np.abs(G.bf(got)[:, :N] - want) <= tol).all() and np.array_equal(got[:, N:], res[:, N:])
    else:
        N = 197 if odd else 200
        wg, wu = bf16((N, K), 1.5 * K ** -0.5, 4), bf16((N, K), K ** -0.5, 5)
        y = G.zeros_bf16(M, N)
        linear(G.dev(x), [G.dev(wg), G.dev(wu)], [], M, K, N, y, _lib.QIE_EPI_SWIGLU)
        (g, gs), (u, us) = products(x, wg), products(x, wu)
        want = u / (1.0 + np.exp(-g)) * g
        tol = 2.0 ** -7 * (np.abs(want) + 1.1 * np.abs(u) * np.abs(g)) + 1e-5 * (1.1 * np.abs(u) * gs + np.abs(g) * us)
        assert (np.abs(G.bf(G.host_bf16(y)) - want) <= tol).all()


@pytest.mark.parametrize("M,K", [(2, 896), (3, 1024), (4, 3584), (5, 2048), (8, 3584), (7, 5120), (8, 5120)])
@pytest.mark.parametrize("num", ["ref", "hf"])
def test_norm_and_keys(qlib, oracle, M, K, num):
    N, eps = 5000, 1e-4 if num == "ref" else 1e-6
    x, nw, w = bf16((M, K), 1.0, 11), bf16((K,), 0.2, 12), bf16((N, K), K ** -0.5, 13)
    nw = oracle.f32_to_bf16(1.0 + G.bf(nw))
    x[0, :K // 2] = 0        # zeros, and a row of small values: the quotient's ranges
    x[1] = oracle.f32_to_bf16(G.bf(x[1]) * np.float32(2.0 ** -60))
    xn = oracle.rmsnorm(x, nw, eps, num)
    y, keys = G.zeros_bf16(M, N), G.dev(np.zeros(M, np.uint64))
    a = _lib.LinearArgsC()
    dx, dw, dn = G.dev(x), G.dev(w), G.dev(nw)
    a.x, a.ldx, a.w[0], a.seg_rows[0], a.M, a.K, a.N = G.p(dx), K, G.p(dw), N, M, K, N
    a.y, a.ldy, a.epilogue, a.numerics, a.norm_w, a.norm_eps = G.p(y), N, _lib.QIE_EPI_STORE, 0 if num == "ref" else 1, G.p(dn), eps
    a.argmax_keys, a.key_col0 = G.p(keys), 0
    G.check(qlib.qie_linear(C.byref(a), None), "qie_linear")
    got = G.host_bf16(y)
    want, scale = products(xn, w)
    # a normed element may round to the neighbouring bf16 (another order of the row's sum of squares): 2^-8 of its share, seldom
    tol = 2.0 ** -7 * np.abs(want) + 1e-3 * scale
    assert (np.abs(G.bf(got) - want) <= tol).all()
    ids = G.zeros((M,), np.int32)
    G.check(qlib.qie_keys_to_ids(G.p(keys), M, G.p(ids), None), "keys")
    assert [int(i) for i in ids.numpy()] == [oracle.argmax(got[m]) for m in range(M)]


@pytest.mark.parametrize("K", [512, 896, 2048, 2560, 3584, 5120])
@pytest.mark.parametrize("num", [0, 1])
def test_fused_norm_is_the_separate_one(qlib, K, num):
    """The norm inside the projection gives qie_rmsnorm's bits, so a row's result does not hang on how many rows share the step."""
    N, eps = 40, 1e-6
    nw, w = bf16((K,), 1.0, 22), bf16((N, K), K ** -0.5, 23)
    dn, dw, xn = G.dev(nw), G.dev(w), G.zeros_bf16(8, K)
    r = np.random.default_rng(K)
    for _ in range(24):   # (an ulp of the root moves one element in 2^15 to another bf16 or so: rows enough to meet some)
        dx = G.dev(G.to_bf16(r.standard_normal((8, K)) * 2.0 ** r.uniform(-6, 6, (8, K))))
        G.check(qlib.qie_rmsnorm(G.p(dx), G.p(dn), G.p(xn), 8, K, eps, num, None), "rmsnorm")
        want = G.zeros((8, N), np.float32)
        linear(xn, [dw], [], 8, K, N, want, _lib.QIE_EPI_F32)
        want = want.numpy()
        for M in range(2, 9):
            y, a = G.zeros((M, N), np.float32), _lib.LinearArgsC()
            a.x, a.ldx, a.w[0], a.seg_rows[0], a.M, a.K, a.N = G.p(dx), K, G.p(dw), N, M, K, N
            a.y, a.ldy, a.epilogue, a.numerics, a.norm_w, a.norm_eps = G.p(y), N, _lib.QIE_EPI_F32, num, G.p(dn), eps
            G.check(qlib.qie_linear(C.byref(a), None), "qie_linear")
            assert np.array_equal(y.numpy(), want[:M]), M


# the sizes where plain rows go back to the skinny kernel, either side of each line
@pytest.mark.parametrize("M,K,N", [(7, 512, 8192), (7, 512, 8193), (8, 512, 130), (2, 640, 130), (3, 1024, 8191), (3, 1024, 8192), (8, 2048, 8192), (5, 2048, 8193)])
def test_lines_to_the_skinny_kernel(qlib, M, K, N):
    x, w = bf16((M, K), 1.0, 31), bf16((N, K), K ** -0.5, 32)
    y = G.zeros_bf16(M, N)
    linear(G.dev(x), [G.dev(w)], [], M, K, N, y, _lib.QIE_EPI_STORE)
    want, scale = products(x, w)
    assert (np.abs(G.bf(G.host_bf16(y)) - want) <= 2.0 ** -8 * np.abs(want) + 1e-5 * scale).all()   # half an ulp of bf16, two orders of one fp32 sum
