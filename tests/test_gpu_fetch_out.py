"""Results by way of a batch's pinned memory (engine.hip fetch_out): sizes that are no multiple of 16 bytes, and more rows than it holds, which
go the other way: the same logits."""
import numpy as np
import pytest

import qwen_inference_engine_amd as q
from qwen_inference_engine_amd import spec as S, weights as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [160, 163])
def test_rows_of_a_layered_step(vocab):
    att = S.LatentAttention(4, 16, 8, 8, 32, 9, 8, 10000.0, 0.2, None)
    spec = S.LayeredSpec("fetch", 64, vocab, 1e-5, (S.LayerSpec(att, S.FeedForward("dense", 96)),), True)
    rng = np.random.default_rng(1)
    tensors = {}
    for n, s in spec.tensor_shapes().items():
        v = np.ones(s, np.float32) if n.endswith(("norm1", "norm2", "final.norm", "dkv.norm")) else \
            (rng.standard_normal(s) / np.sqrt(s[-1] if n != "embed" else 1.0)).astype(np.float32)
        tensors[n] = (np.ascontiguousarray(v).view(np.uint32) >> 16).astype(np.uint16).reshape(s)
    eng = q.Engine(spec, max_ctx=64, dtype="float32").load_tensors(tensors)
    b = eng.batch(2, 64)
    prompt = [int(t) for t in rng.integers(0, vocab, 9)]
    every = b.step([(0, prompt)], range(9))          # more rows than slots
    for want in ([8], [3, 8]):
        b.release(0)
        # (other kernels take the products of fewer rows: fp32 sums in another order)
        assert np.abs(b.step([(0, prompt)], want) - every[want]).max() <= 1e-5 * np.abs(every).max()
    b.close()
    eng.close()


def test_logits_of_an_odd_vocabulary():
    spec = S.tiny("fetch", n_layers=1, hidden=256, n_heads=4, n_kv_heads=2, head_dim=64, ffn=512, vocab=1001)
    eng = q.Engine(spec, device=0, max_ctx=64).init_synthetic(W.SynthParams(seed=3, w_scale=0.08, norm_scale=0.25, bias_scale=0.05))
    one, three = eng.batch(1, 64), eng.batch(3, 64)
    one.prefill(0, [17, 4, 256])
    for m in range(3):
        three.prefill(m, [17, 4, 256])
    want = one.logits()
    assert want.shape == (1, 1001) and want.any()
    assert np.array_equal(three.logits(), np.repeat(want, 3, 0))
    for x in (one, three, eng):
        x.close()


def test_slots_whose_logits_are_more_than_is_pinned():
    """70 slots of 32,000 logits, 9 MB: a few rows by way of the pinned 8 MB, all of them past it."""
    att = S.LatentAttention(4, 16, 8, 8, 32, 9, 8, 10000.0, 0.2, None)
    spec = S.LayeredSpec("fetch", 64, 32000, 1e-5, (S.LayerSpec(att, S.FeedForward("dense", 96)),), True)
    rng = np.random.default_rng(2)
    tensors = {}
    for n, s in spec.tensor_shapes().items():
        v = np.ones(s, np.float32) if n.endswith(("norm1", "norm2", "final.norm", "dkv.norm")) else \
            (rng.standard_normal(s) / np.sqrt(s[-1] if n != "embed" else 1.0)).astype(np.float32)
        tensors[n] = (np.ascontiguousarray(v).view(np.uint32) >> 16).astype(np.uint16).reshape(s)
    eng = q.Engine(spec, max_ctx=64, dtype="float32").load_tensors(tensors)
    b = eng.batch(70, 64)
    toks = [int(t) for t in rng.integers(0, 32000, 70)]
    every = b.step([(m, [t]) for m, t in enumerate(toks)], range(70))
    for m in (0, 41, 69):
        b.release(m)
        one = b.step([(m, [toks[m]])], [0])[0]
        # (other kernels take the products of fewer rows: fp32 sums in another order)
        assert one.any() and np.abs(one - every[m]).max() <= 1e-5 * np.abs(every).max()
    b.close()
    eng.close()
