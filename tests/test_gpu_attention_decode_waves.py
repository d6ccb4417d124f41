"""Decode attention (attn_decode.hpp) where its work changes hands: contexts that end at, before and behind a wave's 32 keys, a step's 128, the one
split of 256 and the one-step splits of 4,096; caches that hold NaN behind the context; few rows and many (fewer splits each), contiguous and
paged; q and the new k already rotated.  Against softmax attention in 64 bits."""
import ctypes as C

import numpy as np
import pytest

import gpu_util as G
from qwen_inference_engine_amd import _lib

pytestmark = pytest.mark.gpu
PREROPED = 0x100   # QIE_ATTN_PREROPED


def attention(q, k, v, G_, hd):
    """q [nq, hd], k / v [nkv, ctx, hd] in 64 bits."""
    kk, vv = np.repeat(k, G_, 0), np.repeat(v, G_, 0)
    s = np.einsum("hd,hkd->hk", q, kk) / np.sqrt(hd)
    p = np.exp(s - s.max(1, keepdims=True))
    return np.einsum("hk,hkd->hd", p / p.sum(1, keepdims=True), vv)


def bf16_words(rng, shape):
    return (rng.standard_normal(shape).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)


@pytest.mark.parametrize("hd,nq,nkv", [(128, 28, 4), (128, 8, 1), (64, 14, 2), (64, 3, 3)])
@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("maxc,ctxs", [(1024, [1, 31, 32]), (1024, [33, 97, 128, 160]), (1024, [255, 256, 257, 384, 385, 1024, 1, 513, 640]),
                                       (4352, [4096]), (4352, [4097, 129, 3000])])
def test_contexts_at_the_edges(qlib, hd, nq, nkv, paged, maxc, ctxs):
    B, L, layer = len(ctxs), 2, 1
    rng = np.random.default_rng(hd + nq + maxc)
    kc, vc = (np.full((B, L, nkv, maxc, hd), 0x7FFF, np.uint16) for _ in range(2))   # NaN wherever no key is
    for m, ctx in enumerate(ctxs):
        kc[m, layer, :, :ctx - 1], vc[m, layer, :, :ctx - 1] = (bf16_words(rng, (nkv, ctx - 1, hd)) for _ in range(2))
    qkv = bf16_words(rng, (B, (nq + 2 * nkv) * hd))
    pos = np.array(ctxs, np.int32) - 1
    cache = _lib.KvCacheC()
    if paged:   # pages of 128 tokens, in another order than the sequences'
        pages = -(-maxc // 128)
        order = rng.permutation(B * pages).astype(np.int32)
        def lay(x):
            out = np.empty((B * pages, L, nkv, 128, hd), np.uint16)
            out[order] = x.reshape(B, L, nkv, pages, 128, hd).transpose(0, 3, 1, 2, 4, 5).reshape(B * pages, L, nkv, 128, hd)
            return out
        dk, dv, table = G.dev(lay(kc)), G.dev(lay(vc)), G.dev(order.reshape(B, pages))
        cache.seq_stride, cache.block_table, cache.page_tokens = L * nkv * 128 * hd, G.p(table), 128
        cache.max_pages = pages
    else:
        dk, dv = G.dev(kc), G.dev(vc)
        cache.seq_stride = L * nkv * maxc * hd
    cache.k, cache.v, cache.n_layers, cache.n_kv_heads, cache.head_dim, cache.max_ctx = G.p(dk), G.p(dv), L, nkv, hd, maxc
    ws, out = G.zeros_bytes(qlib.qie_attention_decode_workspace_bytes(B, nq, nkv, hd, maxc)), G.zeros_bf16(B, nq * hd)
    one = G.dev(np.ones((maxc, hd // 2), np.float32))
    dq, dp = G.dev(qkv), G.dev(pos)
    for _ in range(2):   # the tickets of the first call are zero again
        G.check(qlib.qie_attention_decode(G.p(dq), B, G.p(dp), None, None, G.p(one), G.p(one), nq, C.byref(cache), layer, 1e-6, PREROPED,
                                          G.p(out), G.p(ws), None))
        got = G.bf(G.host_bf16(out)).reshape(B, nq, hd)
        for m, ctx in enumerate(ctxs):
            x = G.bf(qkv[m]).astype(np.float64).reshape(-1, hd)
            k, v = (G.bf(c[m, layer, :, :ctx]).astype(np.float64) for c in (kc, vc))
            k[:, -1], v[:, -1] = x[nq:nq + nkv], x[nq + nkv:]
            want = attention(x[:nq], k, v, nq // nkv, hd)
            # one bf16 rounding of the result; sums of ctx products of 24-bit probabilities (2^-22 of the largest value)
            assert (np.abs(got[m] - want) <= 2.0 ** -8 * np.abs(want) + 2.0 ** -20 * np.abs(v).max()).all(), (ctx, np.abs(got[m] - want).max())


@pytest.mark.parametrize("hd,nq,nkv,maxc", [(128, 28, 4, 1024), (64, 14, 2, 4352)])
def test_calls_of_fewer_rows_share_a_workspace(qlib, hd, nq, nkv, maxc):
    """8, 4, 1 and again 8 rows: the results of fewer rows' splits do not lie in the tickets of the others."""
    rng = np.random.default_rng(hd)
    B, ctxs = 8, [1024, 257, 700, 513, 900, 384, 1000, 640]
    kc, vc = (bf16_words(rng, (B, 1, nkv, maxc, hd)) for _ in range(2))
    dk, dv = G.dev(kc), G.dev(vc)
    cache = _lib.KvCacheC()
    cache.k, cache.v, cache.seq_stride, cache.n_layers, cache.n_kv_heads, cache.head_dim, cache.max_ctx = G.p(dk), G.p(dv), nkv * maxc * hd, 1, nkv, hd, maxc
    ws, one = G.zeros_bytes(qlib.qie_attention_decode_workspace_bytes(B, nq, nkv, hd, maxc)), G.dev(np.ones((maxc, hd // 2), np.float32))
    qkv = bf16_words(rng, (B, (nq + 2 * nkv) * hd))
    dq, dp = G.dev(qkv), G.dev(np.array(ctxs, np.int32) - 1)
    first = None
    for rows in (8, 4, 1, 8, 3, 8):
        out = G.zeros_bf16(B, nq * hd)
        G.check(qlib.qie_attention_decode(G.p(dq), rows, G.p(dp), None, None, G.p(one), G.p(one), nq, C.byref(cache), 0, 1e-6, PREROPED, G.p(out),
                                          G.p(ws), None))
        got = G.bf(G.host_bf16(out)).reshape(B, nq, hd)
        first = got if first is None else first
        # (8 rows may have other splits than fewer: the same sums in another order, one bf16 rounding of each)
        assert (np.abs(got[:rows] - first[:rows]) <= 2.0 ** -7 * np.abs(first[:rows]) + 2.0 ** -20 * 4.0).all(), rows
        assert rows < 8 or np.array_equal(got, first)
    for m, ctx in enumerate(ctxs):
        x = G.bf(qkv[m]).astype(np.float64).reshape(-1, hd)
        k, v = (G.bf(c[m, 0, :, :ctx]).astype(np.float64) for c in (kc, vc))
        k[:, -1], v[:, -1] = x[nq:nq + nkv], x[nq + nkv:]
        want = attention(x[:nq], k, v, nq // nkv, hd)
        assert (np.abs(first[m] - want) <= 2.0 ** -8 * np.abs(want) + 2.0 ** -20 * np.abs(v).max()).all(), ctx


@pytest.mark.parametrize("ctx,masked", [(200, (0, 64)), (700, (128, 384)), (700, (0, 640)), (4096, (0, 3328))])
def test_keys_at_minus_infinity(qlib, ctx, masked):
    """Scores of -inf (keys that hold it, against queries above zero there): a wave's keys, whole splits and every split of the merge's first round
    trip count for nothing."""
    hd, nq, nkv = 64, 14, 2
    rng = np.random.default_rng(ctx)
    kc, vc = (bf16_words(rng, (1, 1, nkv, ctx, hd)) for _ in range(2))
    kc[..., masked[0]:masked[1], 0] = 0xFF80
    qkv = bf16_words(rng, (1, (nq + 2 * nkv) * hd))
    qkv.reshape(-1, hd)[:nq, 0] &= 0x7FFF
    dk, dv = G.dev(kc), G.dev(vc)
    cache = _lib.KvCacheC()
    cache.k, cache.v, cache.seq_stride, cache.n_layers, cache.n_kv_heads, cache.head_dim, cache.max_ctx = G.p(dk), G.p(dv), nkv * ctx * hd, 1, nkv, hd, ctx
    ws, out = G.zeros_bytes(qlib.qie_attention_decode_workspace_bytes(1, nq, nkv, hd, ctx)), G.zeros_bf16(1, nq * hd)
    one = G.dev(np.ones((ctx, hd // 2), np.float32))
    G.check(qlib.qie_attention_decode(G.p(G.dev(qkv)), 1, G.p(G.dev(np.array([ctx - 1], np.int32))), None, None, G.p(one), G.p(one), nq, C.byref(cache),
                                      0, 1e-6, PREROPED, G.p(out), G.p(ws), None))
    x = G.bf(qkv[0]).astype(np.float64).reshape(-1, hd)
    k, v = (G.bf(c[0, 0]).astype(np.float64) for c in (kc, vc))
    k[:, -1], v[:, -1] = x[nq:nq + nkv], x[nq + nkv:]
    want = attention(x[:nq], k, v, nq // nkv, hd)
    got = G.bf(G.host_bf16(out)).reshape(nq, hd)
    assert (np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + 2.0 ** -20 * np.abs(v).max()).all()
