"""The GEMM's tiles of 160 columns (k_gemm_mid.hip) through qie_linear: shapes whose plan takes each of them, in one round of the chip
and in more, with ragged rows and columns; every epilogue (a wave's slice has an odd number of fragments, and the waves' shares of a
k-tile's rows differ); odd columns."""
import numpy as np
import pytest

import gpu_util as G
from gemm_route import routes
from qwen_inference_engine_amd import _lib
from test_gpu_gemm_mid import bf16, linear, products

# rows, columns, K -> tile: each in one round of the chip and in more
SHAPES = [(100, 38002, 512, 8), (129, 37890, 1024, 9), (200, 37891, 1024, 10), (301, 37900, 1024, 11), (65, 58373, 1024, 8), (352, 32835, 512, 9),
          (450, 37890, 2048, 10), (195, 49518, 512, 10), (2856, 6506, 1024, 11)]
EPILOGUE_ROWS, EPILOGUE_K, EPILOGUE_N = [100, 129, 200, 301], 512, 37900


def test_shapes_take_every_wide_tile():
    got = routes([s[:3] for s in SHAPES], f32=True)
    assert [g["tile"] for g in got] == [s[3] for s in SHAPES]
    assert {(g["tile"], g["tiles"] > 256) for g in got} == {(t, more) for t in (8, 9, 10, 11) for more in (False, True)}
    assert not any(g["ahead"] for g in got)
    got = routes([(M, n, EPILOGUE_K) for n in (EPILOGUE_N, EPILOGUE_N + 2) for M in EPILOGUE_ROWS])   # (odd SwiGLU: two weight rows more)
    assert [g["tile"] for g in got] == 2 * [8, 9, 10, 11] and not any(g["ahead"] for g in got)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,tile", SHAPES)
def test_products(qlib, M, N, K, tile):
    x, w = bf16((M, K), 1.0, 1), bf16((N, K), K ** -0.5, 2)
    y = G.zeros((M, N), np.float32)
    linear(G.dev(x), [G.dev(w)], [], M, K, N, y, _lib.QIE_EPI_F32)
    want, scale = products(x, w)
    # two fp32 sums of K products in different orders
    assert (np.abs(y.numpy() - want) <= 1e-5 * scale).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M", EPILOGUE_ROWS)
@pytest.mark.parametrize("epi", ["store", "residual", "swiglu", "swiglu odd"])
def test_epilogues(qlib, oracle, M, epi):
    K, N = EPILOGUE_K, EPILOGUE_N
    x = bf16((M, K), 1.0, 3)
    if epi == "store":
        n = (30000, 5002, 2898)   # the bias changes inside a vector of four columns
        ws, bs = [bf16((r, K), K ** -0.5, 4 + i) for i, r in enumerate(n)], [bf16((r,), 0.5, 7 + i) for i, r in enumerate(n)]
        y = G.zeros_bf16(M, N)
        linear(G.dev(x), [G.dev(w) for w in ws], [G.dev(b) for b in bs], M, K, N, y, _lib.QIE_EPI_STORE)
        want, scale = products(x, np.concatenate(ws))
        want = want + G.bf(np.concatenate(bs))
        G.assert_sum_close(G.host_bf16(y), oracle.f32_to_bf16(want.astype(np.float32)), scale, what=epi)
    elif epi == "residual":
        w, res = bf16((N, K), K ** -0.5, 4), bf16((M, N), 1.0, 5)
        y = G.dev(res)
        linear(G.dev(x), [G.dev(w)], [], M, K, N, y, _lib.QIE_EPI_RESIDUAL)
        acc, scale = products(x, w)
        want = G.bf(res) + G.bf(oracle.f32_to_bf16(acc))
        tol = 2.0 ** -7 * (np.abs(acc) + np.abs(want)) + 1e-5 * scale   # bf16(res + bf16(acc)): an ulp of either rounding
        assert (np.abs(G.bf(G.host_bf16(y)) - want) <= tol).all()
    else:
        N = N // 2 + (1 if epi.endswith("odd") else 0)
        wg, wu = bf16((N, K), 1.5 * K ** -0.5, 4), bf16((N, K), K ** -0.5, 5)
        y = G.zeros_bf16(M, N)
        linear(G.dev(x), [G.dev(wg), G.dev(wu)], [], M, K, N, y, _lib.QIE_EPI_SWIGLU)
        (g, gs), (u, us) = products(x, wg), products(x, wu)
        want = u / (1.0 + np.exp(-g)) * g
        # |silu'| <= 1.1; three bf16 roundings (gate, silu, product) and one of the up sum
        tol = 2.0 ** -7 * (np.abs(want) + 1.1 * np.abs(u) * np.abs(g)) + 1e-5 * (1.1 * np.abs(u) * gs + np.abs(g) * us)
        assert (np.abs(G.bf(G.host_bf16(y)) - want) <= tol).all()
