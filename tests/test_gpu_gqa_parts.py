"""Matrix-core attention whose keys are split into many parts (long contexts, few rows), the parts met in the second pass: value sizes
from half a wave to four rows of one, values turned back by both layouts, tokens one by one, in threes and beside another slot's, against
the fp32 engine's plain attention on the same weights."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# heads, key heads, dim, vdim, layout of values turned back (or none), mask
CASES = [(4, 1, 64, 32, None, "causal"), (4, 4, 32, 64, "halves", "causal"), (8, 2, 64, 96, None, "window"), (4, 1, 128, 128, "interleaved", "causal"),
         (6, 2, 96, 192, None, "causal"), (2, 1, 64, 256, "halves", "causal"), (12, 4, 64, 96, "interleaved", "chunk")]


@pytest.mark.parametrize("heads,kv,dim,vdim,layout,mask", CASES)
def test_parts_meet(heads, kv, dim, vdim, layout, mask):
    import qwen_inference_engine_amd as q
    from qwen_inference_engine_amd import spec as S
    W, V, n = 64, 97, 1125
    rot = dict(rot_dims=vdim if layout else 0, rot_base=100.0, rot_layout=layout or "halves", rot_values=layout is not None)
    if layout:
        dim = vdim   # keys and values turned alike
    a = S.GqaAttention(heads, kv, dim, vdim, dim ** -0.5, qk_norm="weight", mask=mask, mask_size=0 if mask == "causal" else 1100, **rot)
    spec = S.LayeredSpec("parts", W, V, 1e-5, (S.LayerSpec(a, S.FeedForward("dense", 32, act="silu_gated")),), False, block="prenorm")
    rng = np.random.default_rng(heads + dim + vdim)
    T = {}
    for name, shape in spec.tensor_shapes().items():
        v = 1.0 + 0.2 * rng.standard_normal(shape) if "norm" in name else rng.standard_normal(shape) / (np.sqrt(shape[-1]) if name != "embed" else 1.0)
        T[name] = (np.ascontiguousarray(v, dtype=np.float32).view(np.uint32) >> 16).astype(np.uint16).reshape(shape)
    toks = [int(t) for t in rng.integers(0, V, n)]
    out = {}
    for dtype in ("float32", "bfloat16"):
        eng = q.Engine(spec, max_ctx=2304, dtype=dtype).load_tensors(T)
        b = eng.batch(2, 2304, page_tokens=64)
        got = [b.step([(0, toks[:1100])], [1099])]
        for t in range(1100, 1104):
            got.append(b.step([(0, toks[t:t + 1])], [0]))
        got.append(b.step([(0, toks[1104:1107])], range(3)))
        for t in range(1107, 1110):
            got.append(b.step([(0, toks[t:t + 1]), (1, toks[t:t + 1])], [0, 1]))
        got.append(b.step([(0, toks[1110:1125]), (1, toks[:3])], range(18)))   # nearly a whole group of 16 columns
        out[dtype] = np.concatenate(got)
        b.close()
        eng.close()
    want, got = out["float32"], out["bfloat16"]
    # A bf16 rounding is 2^-9 / sqrt(3) = 1.1e-3 of a value on the average; some ten of them stand one behind the other between the embedding and
    # a logit (normed rows, q, k, v, weights of the softmax, heads, activations, the head's rows): 3.6e-3 of a row, three times that for the
    # worst of thirty.  One wrong coordinate in the 128 to 1,152 of a row's heads is 4 to 12 % of its attention.
    err = np.sqrt(((got - want) ** 2).mean(axis=1)) / want.std()
    assert err.max() < 1.1e-2
