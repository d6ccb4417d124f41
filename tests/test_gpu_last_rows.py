"""A prompt's last layer goes on with its last rows alone: the logits of prompts read together and one by one, short and long, on both sides of the
length from which its attention is that of the last rows, are those of the same tokens read but for the last, which a decoding step adds."""
import numpy as np
import pytest

import qwen_inference_engine_amd as q
from qwen_inference_engine_amd import spec as S, weights as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("page", [None, 128])
@pytest.mark.parametrize("length,seqs", [(2, 1), (2, 3), (40, 1), (113, 8), (511, 2), (512, 2), (700, 1)])
def test_last_rows(length, seqs, page):
    spec = S.tiny("last-rows", n_layers=2, hidden=256, n_heads=4, n_kv_heads=2, head_dim=64, ffn=512, vocab=1000)
    eng = q.Engine(spec, device=0, max_ctx=768).init_synthetic(W.SynthParams(seed=3, w_scale=0.08, norm_scale=0.25, bias_scale=0.05))
    rng = np.random.default_rng(length + seqs)
    prompts = [rng.integers(0, 1000, length).tolist() for _ in range(seqs)]
    b = eng.batch(seqs, 768, page_tokens=page)
    b.prefill_batch(0, prompts)
    together = b.logits().copy().view(np.uint16)
    one = eng.batch(1, 768, page_tokens=page)
    f = lambda w: (w.reshape(-1).astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    for z in {0, seqs - 1}:
        one.prefill(0, prompts[z])
        alone = one.logits().copy().view(np.uint16)
        one.prefill(0, prompts[z][:-1])
        one.set_position(0, length - 1, prompts[z][-1])
        one.decode_step()
        stepped = one.logits().copy().view(np.uint16)
        want = f(stepped)
        for got in (together[z], alone):
            # bf16 activations through two layers: 2^-9 a rounding, some ten of them on a row's way
            assert np.linalg.norm(f(got) - want) <= 2.0 ** -6 * np.linalg.norm(want)
    one.close()
    b.close()
    eng.close()
