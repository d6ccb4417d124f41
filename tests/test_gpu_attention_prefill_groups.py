"""Prefill attention by single row groups a wave, in workgroups of 4 and 8 waves, and by pairs of them in workgroups of 2, 4 and 8 (attn_plan.hpp): ragged
rows, waves without a group or a pair, a middle group without a partner, several sequences, pages, NaN in the cache behind the rows; against softmax
attention in 64 bits."""
import ctypes as C

import pytest
import torch

import gpu_util as G
from attn_route import forms
from qwen_inference_engine_amd import _lib

# rows, sequences, heads, key heads, head size, page, (waves of a workgroup, groups of a wave)
CASES = [(33, 1, 14, 2, 64, 0, (4, 1)), (65, 3, 14, 2, 64, 128, (4, 1)), (500, 8, 14, 2, 64, 128, (4, 1)), (49, 2, 7, 7, 128, 0, (4, 1)), (420, 1, 28, 4, 128, 128, (4, 1)),
         (1210, 1, 28, 4, 128, 0, (4, 1)), (301, 8, 28, 4, 128, 0, (8, 1)), (1601, 1, 40, 8, 128, 128, (8, 1)),
         (1100, 1, 14, 2, 64, 0, (2, 2)), (1030, 1, 14, 2, 64, 128, (2, 2)), (250, 4, 14, 2, 64, 128, (2, 2)), (1000, 1, 28, 4, 128, 0, (4, 2)), (1030, 1, 28, 4, 128, 128, (4, 2)),
         (470, 2, 28, 4, 128, 0, (4, 2)), (1801, 1, 28, 4, 128, 128, (8, 2)), (2290, 1, 28, 4, 128, 0, (8, 2)), (950, 2, 28, 4, 128, 128, (8, 2)), (1000, 2, 28, 4, 128, 0, (8, 2))]


def test_cases_take_every_form():
    assert forms([(c[0], c[1], c[2], c[4]) for c in CASES]) == [c[6] for c in CASES]


@pytest.mark.gpu
@pytest.mark.parametrize("R,B,nq,nkv,hd,page,form", CASES)
def test_single_groups(qlib, R, B, nq, nkv, hd, page, form):
    g = torch.Generator().manual_seed(R + B)
    pages = -(-R // page) if page else 0
    room, M = page or R + 70, B * R
    kc, vc = (torch.full((B * pages + 1 if page else B, 1, nkv, room, hd), float("nan"), dtype=torch.bfloat16) for _ in range(2))
    k, v = (torch.randn(B, nkv, R, hd, generator=g).bfloat16() for _ in range(2))
    table = (torch.randperm(B * pages, generator=g).int() + 1).view(B, pages) if page else None
    for c, t in ((kc, k), (vc, v)):
        for b in range(B):
            if page:
                for i in range(pages):
                    n = min(page, R - i * page)
                    c[table[b, i], 0, :, :n] = t[b, :, i * page:i * page + n]
            else:
                c[b, 0, :, :R] = t[b]
    q = torch.randn(M, nq * hd, generator=g).bfloat16()
    dq, dk, dv = (t.cuda() for t in (q, kc, vc))
    pos = torch.arange(R, dtype=torch.int32).repeat(B).cuda()
    out = torch.zeros(M + 1, nq * hd, dtype=torch.bfloat16, device="cuda")
    c = _lib.KvCacheC()
    c.k, c.v, c.seq_stride, c.n_layers, c.n_kv_heads, c.head_dim, c.max_ctx = dk.data_ptr(), dv.data_ptr(), nkv * room * hd, 1, nkv, hd, pages * page if page else room
    if page:
        dt = table.contiguous().cuda()
        c.block_table, c.page_tokens, c.max_pages = dt.data_ptr(), page, pages
    torch.cuda.synchronize()
    G.check(qlib.qie_attention(dq.data_ptr(), M, pos.data_ptr(), R, C.byref(c), 0, nq, out.data_ptr(), None, None))
    torch.cuda.synchronize()
    got = out[:M].double().view(B, R, nq, hd)
    late = torch.ones(R, R, dtype=torch.bool, device="cuda").triu(1)
    for b in range(B):
        for h in range(nq):
            kk, vv = (t[b, h // (nq // nkv)].cuda().double() for t in (k, v))
            s = (dq.view(B, R, nq, hd)[b, :, h].double() @ kk.T) / hd ** 0.5
            want = s.masked_fill(late, float("-inf")).softmax(-1) @ vv
            # one bf16 rounding of the result; probabilities of 16 bits and more (2^-16 of the largest value)
            assert ((got[b, :, h] - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -14 * vv.abs().max()).all(), (b, h)
    assert not out[M].any()
