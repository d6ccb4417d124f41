"""Attention of prompts of less than 32 rows (prompt_attention, what a prompt's layers call): on the matrix cores, probabilities of 24 bits; against
softmax attention in 64 bits and, beside it, the general kernel's distance from that.  One row group and two, several sequences, pages, NaN behind the rows."""
import ctypes as C

import pytest
import torch

import gpu_util as G
from qwen_inference_engine_amd import _lib

pytestmark = pytest.mark.gpu
SYMBOL = "_ZN3qie16prompt_attentionEPKvlPKiiPK12qie_kv_cacheiiPvS7_P12ihipStream_t"


@pytest.mark.parametrize("R,B,nq,nkv,hd,page", [(1, 3, 14, 2, 64, 0), (2, 1, 14, 2, 64, 0), (15, 2, 7, 7, 128, 0), (16, 1, 28, 4, 128, 128), (17, 5, 14, 2, 64, 128),
                                                (24, 1, 14, 2, 64, 0), (31, 40, 28, 4, 128, 0), (32, 1, 14, 2, 64, 0)])
def test_short_prompts(qlib, R, B, nq, nkv, hd, page):
    g = torch.Generator().manual_seed(R + B)
    room, M = page or R + 70, B * R
    shape = (B + 1, 1, nkv, room, hd) if page else (B, 1, nkv, room, hd)
    table = (torch.randperm(B, generator=g).int() + 1) if page else torch.arange(B).int()
    kc, vc = (torch.full(shape, float("nan"), dtype=torch.bfloat16) for _ in range(2))
    for c in (kc, vc):
        for b in range(B):
            c[table[b], 0, :, :R] = torch.randn(nkv, R, hd, generator=g).bfloat16()
    q = torch.randn(M, nq * hd, generator=g).bfloat16()
    dq, dk, dv, dt = (t.cuda() for t in (q, kc, vc, table))
    pos = torch.arange(R, dtype=torch.int32).repeat(B).cuda()
    c = _lib.KvCacheC()
    c.k, c.v, c.seq_stride, c.n_layers, c.n_kv_heads, c.head_dim, c.max_ctx = dk.data_ptr(), dv.data_ptr(), nkv * room * hd, 1, nkv, hd, room
    if page:
        c.block_table, c.page_tokens, c.max_pages = dt.data_ptr(), page, 1
    ws = torch.zeros(max(16, qlib.qie_attention_workspace_bytes(M, nq, hd, room)), dtype=torch.uint8, device="cuda")
    fn = getattr(C.CDLL(_lib.load()._name), SYMBOL)
    fn.restype, fn.argtypes = C.c_int, [C.c_void_p, C.c_int64, C.c_void_p, C.c_int32, C.c_void_p, C.c_int32, C.c_int32, C.c_void_p, C.c_void_p, C.c_void_p]
    torch.cuda.synchronize()
    got = []
    for call in (fn, qlib.qie_attention):
        out = torch.zeros(M + 1, nq * hd, dtype=torch.bfloat16, device="cuda")
        torch.cuda.synchronize()
        G.check(call(dq.data_ptr(), M, pos.data_ptr(), R, C.byref(c), 0, nq, out.data_ptr(), ws.data_ptr(), None))
        torch.cuda.synchronize()
        assert not out[M].any()
        got.append(out[:M].view(B, R, nq, hd))
    late = torch.ones(R, R, dtype=torch.bool, device="cuda").triu(1)
    off = [0, 0]   # results that are not the bf16 nearest to the exact ones
    for b in range(B):
        for h in range(nq):
            k, v = (t[int(table[b]), 0, h // (nq // nkv), :R].double() for t in (dk, dv))
            s = (dq.view(B, R, nq, hd)[b, :, h].double() @ k.T) / hd ** 0.5
            want = s.masked_fill(late, float("-inf")).softmax(-1) @ v
            for i, o in enumerate(got):
                err = (o[b, :, h].double() - want).abs()
                # one bf16 rounding, and fp32 sums of at most 31 products and hd of a score
                assert (err <= 2.0 ** -8 * want.abs() * (1 + 2.0 ** -10) + 2.0 ** -18 * v.abs().max()).all(), (i, b, h)
                off[i] += int((o[b, :, h] != want.bfloat16()).sum())
    assert off[0] <= 1.5 * off[1] + 20   # of some hundred to 100,000 values; two fp32 orders differ by less
