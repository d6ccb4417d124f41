"""Steps whose delta rules all walk their rows in order make no pieces, nor room for the pieces' states."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_walks_need_no_pieces():
    import qwen_inference_engine_amd as q
    from qwen_inference_engine_amd import spec as S
    V, slots = 97, 56
    spec = S.LayeredSpec("walks", 64, V, 1e-5, (S.LayerSpec(S.GatedDelta(16, 8, 128, 128, 4), S.FeedForward("dense", 32, act="silu_gated")),), False, block="prenorm")
    rng = np.random.default_rng(0)
    T = {n: (np.ascontiguousarray(rng.standard_normal(s) * s[-1] ** -0.5, dtype=np.float32).view(np.uint32) >> 16).astype(np.uint16).reshape(s)
         for n, s in spec.tensor_shapes().items()}
    eng = q.Engine(spec, max_ctx=2048, dtype="bfloat16").load_tensors(T)
    b = eng.batch(slots, 2048, page_tokens=64)

    def step(n, rows):
        for m in range(slots):
            b.release(m)
        for _ in range(2):   # (the second: nothing is made for the first time)
            b.step([(m, rng.integers(0, V, rows // 2)) for m in range(n)], [0])
        torch.cuda.synchronize()
        return torch.cuda.mem_get_info()[0]
    # the same rows: 56 entries of 128 and 8 of 896 (112 pieces of 64 rows have states of 350 MB)
    assert abs(step(56, 256) - step(8, 1792)) < 16 << 20
    b.close()
    eng.close()
