"""fp8 projections of long plain rows, up to 8 rows of X (k_decode_fp8.hip dec8s_kernel): uneven shares of K, a block's second tile, either
layout of the weights, every epilogue, either number of X rows that a chunk carries; and weights in several segments, which it leaves to others."""
import ctypes as C

import numpy as np
import pytest

import gpu_util as G
from qwen_inference_engine_amd import _lib
from test_gpu_fp8 import _fp8_dev, _tiled
from test_gpu_ops import _abs_scale, _linear, rand_bf16

pytestmark = pytest.mark.gpu


# rows, K, columns (tests/test_fp8_long_rule.py holds the dispatch to this kernel for them)
SHAPES = [(1, 2176, 3072), (3, 2176, 4112), (4, 3712, 3088), (5, 2176, 4112), (8, 2176, 8208), (8, 18944, 3584)]


@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("M,K,N", SHAPES)
def test_long_rows(oracle, qlib, M, K, N, tiled):
    if M == 1 and not tiled:
        pytest.skip("one row of plain weights is the row GEMV's")
    x = rand_bf16(oracle, (M, K), seed=M + K)
    d, dq = _fp8_dev(qlib, rand_bf16(oracle, (N, K), 0.05, seed=N))
    w = [(_tiled(qlib, d, N, K) if tiled else d, N)]
    flags = _lib.QIE_LINEAR_FP8 | (_lib.QIE_LINEAR_FP8_T16 if tiled else 0)
    ldy, scale = N + 7, _abs_scale(oracle, x, dq)
    exact = oracle.bf16_to_f32(x).astype(np.float64) @ oracle.bf16_to_f32(dq).astype(np.float64).T

    def run(epi, y0, **kw):
        y = G.dev(y0.copy())
        _linear(qlib, G.dev(x), w, kw.pop("biases", []), M, K, N, y, epi, ldy=ldy, flags=flags, **kw)
        return y

    # fp32: a chain of at most 320 products in each of a wave's 8 sums, 6 meetings in pairs; 1e-5 of the absolute sum is the repository's bound
    y = G.host(run(_lib.QIE_EPI_F32, np.full((M, ldy), 3.0, np.float32)))
    assert (np.abs(y[:, :N] - exact) <= 1e-5 * scale).all() and (y[:, N:] == 3.0).all()
    res = rand_bf16(oracle, (M, ldy), seed=5)
    y = G.host_bf16(run(_lib.QIE_EPI_RESIDUAL, res))
    want = oracle.f32_to_bf16((oracle.bf16_to_f32(res[:, :N]) + oracle.bf16_to_f32(oracle.matmul(x, dq))).astype(np.float32))
    # (a last bit of the product, and of the sum it goes into)
    ulp = 2.0 ** -7 * (np.abs(exact) + np.abs(oracle.bf16_to_f32(want).astype(np.float64)))
    diff = np.abs(oracle.bf16_to_f32(y[:, :N]).astype(np.float64) - oracle.bf16_to_f32(want))
    assert (diff <= np.maximum(ulp, 1e-5 * scale)).all() and np.array_equal(y[:, N:], res[:, N:])
    b = rand_bf16(oracle, (N,), 0.1, seed=9)
    keys = G.dev(np.zeros(M, np.uint64))
    y = G.host_bf16(run(_lib.QIE_EPI_STORE, res, biases=[G.dev(b)], keys=keys))
    G.assert_sum_close(y[:, :N], oracle.matmul(x, dq, b), scale, what=f"M={M} K={K} N={N}")
    ids = G.zeros((M,), np.int32)
    G.check(qlib.qie_keys_to_ids(G.p(keys), M, G.p(ids), None))
    for m in range(M):
        assert G.host(ids)[m] == oracle.argmax(np.ascontiguousarray(y[m, :N]))


@pytest.mark.parametrize("K,N,bound", [(5120, 4096, 8.5e-8), (18944, 3584, 1.0e-7)])
def test_sums_are_short(oracle, qlib, K, N, bound):
    """The sums of a long row are many short ones that meet in pairs.  A rounding of a partial sum that holds the share s of the products
    costs 0.41 * 2^-24 * sqrt(s) of the result on the average, and they add up in squares: 8 chains of K / 8,192 chunks a wave, 3 steps
    of pairs there and 3 between the waves: 7 such units at K = 5,120, 11 at 18,944, 6.5e-8 and 8.1e-8; a chain over a wave's share has
    14 and 42."""
    M = 8
    x = rand_bf16(oracle, (M, K), seed=1)
    d, dq = _fp8_dev(qlib, rand_bf16(oracle, (N, K), 0.05, seed=2))
    exact = oracle.bf16_to_f32(x).astype(np.float64) @ oracle.bf16_to_f32(dq).astype(np.float64).T
    y = G.zeros((M, N), np.float32)
    _linear(qlib, G.dev(x), [(_tiled(qlib, d, N, K), N)], [], M, K, N, y, _lib.QIE_EPI_F32, flags=_lib.QIE_LINEAR_FP8 | _lib.QIE_LINEAR_FP8_T16)
    err = np.linalg.norm(G.host(y) - exact) / np.linalg.norm(exact)
    assert err < bound


@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("M,K,r", [(2, 2176, (2048, 0, 1536)), (8, 2176, (2048, 0, 1536)), (2, 2176, (2048, 1024, 512)), (2, 2176, (0, 0, 3584)),
                                   (8, 2176, (1024, 0, 512)), (2, 3584, (1024, 0, 512)), (2, 3584, (0, 0, 1536)), (2, 3584, (0, 1536, 0))])
def test_weights_in_several_segments(oracle, qlib, M, K, r, tiled):
    """Columns take weights, scales and biases of their own segment, whichever segments there are."""
    N = sum(r)
    x, res = rand_bf16(oracle, (M, K), seed=M), rand_bf16(oracle, (M, N), seed=5)
    wf, b = rand_bf16(oracle, (N, K), 0.05, seed=N), rand_bf16(oracle, (N,), 0.1, seed=9)
    at = np.concatenate([[0], np.cumsum(r)])
    scale = np.repeat(np.float32([1.0, 2.0, 4.0]), r)   # segments of unlike size: unlike row scales
    wf = oracle.f32_to_bf16(oracle.bf16_to_f32(wf) * scale[:, None])
    parts = [_fp8_dev(qlib, wf[at[i]:at[i + 1]].copy()) if n else None for i, n in enumerate(r)]
    dq = np.concatenate([p[1] for p in parts if p])
    w = [(_tiled(qlib, p[0], n, K) if tiled else p[0]) if p else None for p, n in zip(parts, r)]
    other = _fp8_dev(qlib, rand_bf16(oracle, (N, K), 1.0, seed=N + 1))[0]
    flags = _lib.QIE_LINEAR_FP8 | (_lib.QIE_LINEAR_FP8_T16 if tiled else 0)

    def run(epi, biases):
        y = G.dev(res.copy())
        a = _lib.LinearArgsC()
        dx = G.dev(x)
        a.x, a.ldx, a.M, a.K, a.N, a.y, a.ldy, a.epilogue, a.flags = G.p(dx), K, M, K, N, G.p(y), N, epi, flags
        a.w[0] = G.p(other)   # (an empty first segment still has an address, here of as many rows that are not to be read)
        for i in range(3):
            if r[i]:
                a.w[i], a.seg_rows[i] = G.p(w[i]), r[i]
            if r[i] and biases:
                a.bias[i] = G.p(biases[i])
        G.check(qlib.qie_linear(C.byref(a), None), "qie_linear")
        return G.host_bf16(y)

    size = _abs_scale(oracle, x, dq)
    y = run(_lib.QIE_EPI_STORE, [G.dev(b[at[i]:at[i + 1]].copy()) if r[i] else None for i in range(3)])
    G.assert_sum_close(y, oracle.matmul(x, dq, b), size, what="store")
    got = oracle.bf16_to_f32(run(_lib.QIE_EPI_RESIDUAL, None)).astype(np.float64)
    prod = oracle.bf16_to_f32(oracle.matmul(x, dq)).astype(np.float64)
    want = oracle.bf16_to_f32(res) + prod
    # a last bit of the product, and of the sum it goes into
    assert (np.abs(got - want) <= np.maximum(2.0 ** -7 * (np.abs(prod) + np.abs(want)), 1e-5 * size)).all()


def test_a_row_does_not_depend_on_its_neighbours(oracle, qlib):
    K, N = 2176, 3072
    x = rand_bf16(oracle, (8, K), seed=3)
    w = _tiled(qlib, _fp8_dev(qlib, rand_bf16(oracle, (N, K), 0.05, seed=4))[0], N, K)
    rows = []
    for M in (1, 4, 8):
        y = G.zeros((M, N), np.float32)
        _linear(qlib, G.dev(x[:M].copy()), [(w, N)], [], M, K, N, y, _lib.QIE_EPI_F32, flags=_lib.QIE_LINEAR_FP8 | _lib.QIE_LINEAR_FP8_T16)
        rows.append(G.host(y))
    assert np.array_equal(rows[0], rows[2][:1]) and np.array_equal(rows[1], rows[2][:4])
