"""Prefill attention of few rows and of many, one sequence and several (attn_plan.hpp: workgroups by the rows, heads and sequences of a call): ragged
rows, waves without rows, NaN in the cache behind the rows; against softmax attention in 64 bits."""
import ctypes as C

import pytest
import torch

import gpu_util as G
from attn_route import forms
from qwen_inference_engine_amd import _lib

# rows, sequences, heads, key heads, head size
CASES = [(32, 1, 14, 2, 64), (113, 2, 14, 2, 64), (301, 1, 28, 4, 128), (449, 1, 7, 7, 128), (620, 1, 28, 4, 128), (1310, 1, 28, 4, 128), (301, 8, 28, 4, 128)]


def test_forms():
    """Single groups in 4 waves and, beyond one round of the chip, in 8 (pairs: test_gpu_attention_prefill_groups.py)."""
    assert forms([(R, B, nq, hd) for R, B, nq, nkv, hd in CASES]) == [(4, 1)] * 6 + [(8, 1)]


@pytest.mark.gpu
@pytest.mark.parametrize("R,B,nq,nkv,hd", CASES)
def test_rows_of_every_workgroup(qlib, R, B, nq, nkv, hd):
    g = torch.Generator().manual_seed(R + B)
    room, M = R + 70, B * R
    kc, vc = (torch.full((B, 1, nkv, room, hd), float("nan"), dtype=torch.bfloat16) for _ in range(2))
    for c in (kc, vc):
        c[:, 0, :, :R] = torch.randn(B, nkv, R, hd, generator=g).bfloat16()
    q = torch.randn(M, nq * hd, generator=g).bfloat16()
    dq, dk, dv = (t.cuda() for t in (q, kc, vc))
    pos = torch.arange(R, dtype=torch.int32).repeat(B).cuda()
    out = torch.zeros(M + 1, nq * hd, dtype=torch.bfloat16, device="cuda")
    c = _lib.KvCacheC()
    c.k, c.v, c.seq_stride, c.n_layers, c.n_kv_heads, c.head_dim, c.max_ctx = dk.data_ptr(), dv.data_ptr(), nkv * room * hd, 1, nkv, hd, room
    torch.cuda.synchronize()
    G.check(qlib.qie_attention(dq.data_ptr(), M, pos.data_ptr(), R, C.byref(c), 0, nq, out.data_ptr(), None, None))
    torch.cuda.synchronize()
    got = out[:M].double().view(B, R, nq, hd)
    late = torch.ones(R, R, dtype=torch.bool, device="cuda").triu(1)
    for b in range(B):
        for h in range(nq):
            k, v = (t[b, 0, h // (nq // nkv), :R].double() for t in (dk, dv))
            s = (dq.view(B, R, nq, hd)[b, :, h].double() @ k.T) / hd ** 0.5
            want = s.masked_fill(late, float("-inf")).softmax(-1) @ v
            # one bf16 rounding of the result; probabilities of 16 bits and more (2^-16 of the largest value)
            assert ((got[b, :, h] - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -14 * v.abs().max()).all(), (b, h)
    assert not out[M].any()
