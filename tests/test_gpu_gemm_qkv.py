"""The QKV product whose epilogue turns q and k and writes the cache (gemm_qkv, what a prompt's layers call) against the product and
qie_qkv_post: the same bits.  Every form of k_gemm_few.hip, every tile of k_gemm_mid.hip and the 256x256 kernel, split and whole, ragged rows, several prompts
in a tile, heads of 8, 64 and 128, contiguous and paged; and a K that no kernel with that epilogue takes."""
import ctypes as C

import numpy as np
import pytest
import torch

import gpu_util as G
from gemm_route import routes
from qwen_inference_engine_amd import _lib
from qwen_inference_engine_amd._lib import KvCacheC, LinearArgsC

SYMBOL = "_ZN3qie8gemm_qkvEPK15qie_linear_argsPK12qie_kv_cacheiiPKfPtP12ihipStream_tPb"


# heads, key heads, head size, K, rows of a prompt, prompts, page, tile (k_gemm_mid.hip's, "few 0" ..: k_gemm_few.hip's forms, -1: the 256x256 kernel,
# None: one without this epilogue)
CASES = [
    (14, 2, 64, 896, 17, 1, 0, "few 0"), (14, 2, 64, 896, 113, 1, 128, "few 1"), (14, 2, 64, 896, 37, 5, 128, "few 1"),
    (28, 4, 128, 3584, 71, 1, 128, "few 2"), (28, 4, 128, 3584, 31, 3, 0, "few 2"), (14, 2, 64, 896, 301, 1, 0, "few 3"),
    (14, 2, 64, 896, 79, 5, 128, "few 3"), (28, 4, 128, 3584, 183, 1, 128, "few 4"), (28, 4, 128, 3584, 61, 3, 0, "few 4"),
    (14, 2, 64, 896, 507, 1, 128, 0), (14, 2, 64, 256, 75, 4, 0, 0), (2, 1, 64, 2048, 601, 1, 128, 0), (2, 1, 64, 12288, 70, 3, 0, 0),
    (14, 2, 64, 896, 1501, 1, 0, 1), (28, 4, 128, 3584, 63, 1, 128, 0), (28, 4, 128, 3584, 301, 1, 0, 2),
    (28, 4, 128, 3584, 1030, 1, 128, 4), (28, 4, 128, 512, 2100, 2, 256, -1), (28, 4, 128, 512, 1363, 3, 0, -1),
    (3, 1, 8, 256, 65, 2, 0, 0), (14, 2, 64, 928, 300, 1, 0, None), (28, 4, 128, 3584, 2500, 1, 0, -1), (28, 4, 128, 3584, 2048, 1, 128, 7),
    (28, 4, 128, 3584, 1024, 8, 128, 11), (28, 4, 128, 3584, 4096, 1, 0, 10), (28, 4, 128, 3584, 1363, 1, 128, 5), (14, 2, 64, 896, 2300, 1, 0, 3),
    (14, 2, 64, 896, 6000, 1, 0, 9), (16, 4, 128, 256, 1540, 1, 0, 6), (56, 8, 128, 256, 195, 1, 128, 8), (56, 8, 128, 4096, 67, 1, 0, 3),
    (32, 8, 128, 16384, 500, 2, 128, -1)]


def test_cases_take_every_kernel_with_the_epilogue():
    got = routes([(c[4] * c[5], (c[0] + 2 * c[1]) * c[2], c[3], 0, c[0] * c[2] % 64 != 0 or c[1] * c[2] % 64 != 0) for c in CASES])
    for c, r in zip(CASES, got):
        if c[7] is None:
            assert c[3] % 64 != 0, c
        else:
            assert ("few %d" % r["few"] if r["few"] >= 0 else r["tile"]) == c[7] and (c[7] != -1 or r["parts"] >= 1), (c, r)
    assert {r["tile"] for r in got} == set(range(-2, 12)) and {r["few"] for r in got} == set(range(-1, 5))
    assert {r["parts"] for r, c in zip(got, CASES) if c[7] == -1} >= {1, 2}   # the 256x256 kernel whole and split
    assert {r["splitk"] > 1 for r in got if r["tile"] == 0} == {False, True}


@pytest.mark.gpu
@pytest.mark.parametrize("nq,nkv,hd,K,n,seqs,page,tile", CASES)
def test_as_the_product_and_its_post_pass(qlib, nq, nkv, hd, K, n, seqs, page, tile):
    M, QD, KD, ctx, layers, layer = n * seqs, nq * hd, nkv * hd, n + 3, 2, 1
    N = QD + 2 * KD
    g = torch.Generator("cuda").manual_seed(M + K)

    def t(*shape, scale=1.0):
        return (torch.randn(*shape, generator=g, device="cuda") * scale).bfloat16()
    x, ws, bs = t(M, K), [t(r, K, scale=K ** -0.5) for r in (QD, KD, KD)], [t(r) for r in (QD, KD, KD)]
    ang = torch.arange(ctx, device="cuda")[:, None] * 1e4 ** (-torch.arange(hd // 2, device="cuda") / (hd // 2))
    cs, sn = ang.cos().float().contiguous(), ang.sin().float().contiguous()
    turns = torch.stack([cs, sn], -1).contiguous()
    pos = torch.arange(M, device="cuda", dtype=torch.int32) % n
    pages = -(-ctx // page) if page else 0
    table = (torch.randperm(seqs * pages, generator=g, device="cuda").int() + 1) if page else None

    def cache():
        c = KvCacheC()
        shape = (seqs * pages + 1, layers, nkv, page, hd) if page else (seqs, layers, nkv, ctx, hd)
        kv = [torch.full(shape, 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
        c.k, c.v, c.seq_stride = kv[0].data_ptr(), kv[1].data_ptr(), kv[0][0].numel()
        c.n_layers, c.n_kv_heads, c.head_dim, c.max_ctx = layers, nkv, hd, ctx
        if page:
            c.block_table, c.page_tokens, c.max_pages = table.data_ptr(), page, pages
        return c, kv

    def args(y):
        a = LinearArgsC()
        a.x, a.ldx, a.M, a.K, a.N, a.y, a.ldy, a.epilogue = x.data_ptr(), K, M, K, N, y.data_ptr(), N, _lib.QIE_EPI_STORE
        for i, (w, b) in enumerate(zip(ws, bs)):
            a.w[i], a.bias[i], a.seg_rows[i] = w.data_ptr(), b.data_ptr(), w.shape[0]
        return a
    y, q = torch.zeros(M, N, dtype=torch.bfloat16, device="cuda"), torch.zeros(M, QD, dtype=torch.bfloat16, device="cuda")
    c, kv = cache()
    torch.cuda.synchronize()
    G.check(qlib.qie_linear(C.byref(args(y)), None), "qie_linear")
    G.check(qlib.qie_qkv_post(y.data_ptr(), M, pos.data_ptr(), n, None, None, cs.data_ptr(), sn.data_ptr(), nq, C.byref(c), layer, 1e-6,
                              _lib.QIE_NUMERICS_REF, q.data_ptr(), None), "qie_qkv_post")
    fn = getattr(C.CDLL(_lib.load()._name), SYMBOL)
    fn.restype = C.c_int
    fn.argtypes = [C.c_void_p, C.c_void_p, C.c_int32, C.c_int32] + [C.c_void_p] * 4
    y2, q2, done = torch.zeros_like(y), torch.full_like(q, 7.0), C.c_bool()
    c2, kv2 = cache()
    torch.cuda.synchronize()
    G.check(fn(C.byref(args(y2)), C.byref(c2), layer, n, turns.data_ptr(), q2.data_ptr(), None, C.byref(done)), "gemm_qkv")
    torch.cuda.synchronize()
    assert done.value == (tile is not None)
    if tile is None:
        assert torch.equal(y, y2) and (q2 == 7.0).all()
        return
    assert torch.equal(q, q2)
    for a, b in zip(kv, kv2):   # untouched: the other layer, the rest of the context and the page that nobody holds
        assert torch.equal(a, b)
    assert np.isfinite(q2.float().sum().item())
