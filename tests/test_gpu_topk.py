"""The radix selection of top-k sampling (k_sampling.hip) at the sizes where it can go wrong: fewer logits than k, one more and one
less than a slice, every merge width, rows of equal values, of masked (-inf) and NaN values, negative rows; against the oracle."""
import ctypes as C

import numpy as np
import pytest

import gpu_util as G
from qwen_inference_engine_amd._lib import SamplingC

pytestmark = pytest.mark.gpu


def sampled(qlib, lg, k, T, tp, seed, step):
    M, V = lg.shape
    s = SamplingC()
    s.top_k, s.temperature, s.top_p, s.seed = k, T, tp, seed
    ids, ws = G.zeros((M,), np.int32), G.zeros_bytes(qlib.qie_sample_workspace_bytes(M, V))
    G.check(qlib.qie_sample(G.p(G.dev(lg)), M, V, V, C.byref(s), G.p(G.dev(np.asarray(step, np.int32))), G.p(ids), G.p(ws), None))
    return [int(i) for i in G.host(ids)]


@pytest.mark.parametrize("V,k", [(3, 2), (3, 50), (40, 50), (50, 50), (4095, 256), (4096, 63), (4097, 64), (8193, 65), (33000, 255), (152064, 256),
                                 (200000, 256)])
def test_widths(qlib, oracle, V, k):
    r = np.random.default_rng(V + k)
    lg = oracle.f32_to_bf16((r.standard_normal((3, V)) * 2 - [[0.0], [9.0], [0.0]]).astype(np.float32))   # a row of negative values
    lg[2] = oracle.f32_to_bf16(r.integers(0, 3, V).astype(np.float32))                                     # thousands of ties
    for T, tp, seed in ((0.7, 1.0, 1234), (1.5, 0.8, 99)):
        assert sampled(qlib, lg, k, T, tp, seed, [0, 5, 9]) == [oracle.sample(lg[m], k, T, tp, seed + st) for m, st in enumerate((0, 5, 9))]


@pytest.mark.parametrize("V", [30, 5000, 152064])
def test_masked_rows(qlib, oracle, V):
    r = np.random.default_rng(V)
    f = (r.standard_normal((4, V)) * 2).astype(np.float32)
    f[0, r.permutation(V)[20:]] = -np.inf    # 20 candidates left
    f[1] = -np.inf
    f[1, V // 2] = -3.0                      # one
    f[2] = -7.0                              # all equal
    f[3, ::3] = np.nan                       # NaN is no candidate
    lg = oracle.f32_to_bf16(f)
    assert sampled(qlib, lg, 50, 0.9, 0.95, 7, [0, 1, 2, 3]) == [oracle.sample(lg[m], 50, 0.9, 0.95, 7 + m) for m in range(4)]
    lg = np.full((1, V), 0xFF80, np.uint16)  # nothing to choose from
    assert sampled(qlib, lg, 50, 0.9, 0.95, 7, [0]) == [-1]


@pytest.mark.parametrize("V,k", [(8192, 2), (20000, 50), (152064, 50), (152064, 256)])
def test_where_the_best_are(qlib, oracle, V, k):
    """Few candidates over the slices' bound and more than are put in order at once: the best spread out, at the end, in one slice, in every 4th."""
    r = np.random.default_rng(V * k)
    f = (r.standard_normal((4, V)) * 2).astype(np.float32)
    f[1] = np.arange(V) * np.float32(30.0 / V)
    f[2, 4096:8192] += 20.0
    f[3, (np.arange(V) // 4096) % 4 != 0] -= 20.0
    lg = oracle.f32_to_bf16(f)
    for T, tp, seed in ((0.7, 0.9, 3), (2.5, 1.0, 4)):
        assert sampled(qlib, lg, k, T, tp, seed, [0, 1, 2, 3]) == [oracle.sample(lg[m], k, T, tp, seed + m) for m in range(4)]
