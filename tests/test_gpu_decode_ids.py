"""Ids of several decode steps fetched at once, after positions set one behind the other without a wait: equal to step by step, and to
the history, on ragged slots with one of them idle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 3, 8])
def test_ids_equal_step_by_step(batch):
    import qwen_inference_engine_amd as q
    from qwen_inference_engine_amd import spec as S, weights as W
    spec = S.tiny("ids", n_layers=2, hidden=256, n_heads=4, n_kv_heads=2, head_dim=64, ffn=512, vocab=1000)
    eng = q.Engine(spec, device=0, max_ctx=128).init_synthetic(W.SynthParams(seed=3, w_scale=0.08, norm_scale=0.25, bias_scale=0.05))
    b = eng.batch(batch, 128)
    live = [m for m in range(batch) if batch == 1 or m != 1]
    rng = np.random.default_rng(1)
    prompts = {m: rng.integers(0, 1000, 9 + 5 * m).tolist() for m in live}
    for m in live:
        b.prefill(m, prompts[m])
    out = []
    for many in (False, True, True):
        for m in live:
            b.set_position(m, len(prompts[m]), 7 + m)
        out.append(np.stack([b.decode_step() for _ in range(12)]) if not many else b.decode(12))
        for m in live:
            assert b.history(m, len(prompts[m]) + 13)[len(prompts[m]):].tolist() == [7 + m] + out[-1][:, m].tolist()
    assert (out[0][:, live] == out[1][:, live]).all() and (out[1][:, live] == out[2][:, live]).all()
    assert b.decode(0).shape == (0, batch)
    b.close()
    eng.close()


def test_more_ids_than_are_fetched_at_once():
    """A call of more ids than the pinned room takes gives those of calls that fit it."""
    import qwen_inference_engine_amd as q
    from qwen_inference_engine_amd import spec as S, weights as W
    spec = S.tiny("ids", n_layers=1, hidden=128, n_heads=2, n_kv_heads=1, head_dim=64, ffn=256, vocab=500)
    eng = q.Engine(spec, device=0, max_ctx=2304).init_synthetic(W.SynthParams(seed=3, w_scale=0.08, norm_scale=0.25, bias_scale=0.05))
    b = eng.batch(8, 2304)
    for m in range(8):
        b.prefill(m, list(range(5 + m)))
    out = []
    for parts in ((800, 800, 550), (2150,)):   # 17,200 ids in all
        for m in range(8):
            b.set_position(m, 5 + m, 7 + m)
        out.append(np.concatenate([b.decode(n) for n in parts]))
    assert np.array_equal(out[0], out[1])
    assert b.history(7, 12 + 2151)[13:].tolist() == out[1][:, 7].tolist()
    b.close()
    eng.close()
