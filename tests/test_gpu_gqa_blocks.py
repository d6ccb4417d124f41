"""Matrix-core attention of prompts: blocks of keys that a group of 16 rows sees whole, in part and not at all, under every mask and score, pages of one
block and of more, whole chains of blocks and parts of them, against the fp32 engine's plain attention on the same weights."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# heads, key heads, dim = vdim, options; four heads of a key head share its tiles, others load for themselves
CASES = [(4, 1, 128, dict(softcap=5.0)), (8, 2, 64, dict(mask="window", mask_size=40, mask_keep=37)), (4, 1, 64, dict(mask="window", mask_size=33)),
         (4, 1, 96, dict(mask="chunk", mask_size=48, softcap=20.0)), (4, 1, 64, dict(weights="sigmoid")), (4, 1, 192, dict(slope_bias=True, sink=True)),
         (4, 1, 256, dict(dist_bias=True)), (6, 2, 64, dict(softcap=5.0)), (6, 2, 128, dict(mask="window", mask_size=40, mask_keep=37)), (2, 2, 64, dict(weights="sigmoid"))]


@pytest.mark.parametrize("page", [32, 64])
@pytest.mark.parametrize("heads,kv,dim,more", CASES)
def test_blocks(heads, kv, dim, more, page):
    import qwen_inference_engine_amd as q
    from qwen_inference_engine_amd import spec as S
    W, V = 64, 97
    a = S.GqaAttention(heads, kv, dim, dim, dim ** -0.5, qk_norm="weight", **more)
    spec = S.LayeredSpec("blocks", W, V, 1e-5, (S.LayerSpec(a, S.FeedForward("dense", 32, act="silu_gated")),), False, block="prenorm")
    rng = np.random.default_rng(heads + dim)
    T = {}
    for name, shape in spec.tensor_shapes().items():
        v = 1.0 + 0.2 * rng.standard_normal(shape) if "norm" in name else rng.standard_normal(shape) / (np.sqrt(shape[-1]) if name != "embed" else 1.0)
        if name.endswith((".r1", ".r2")):   # (ln(1 + r2 distance))
            v = np.abs(v)
        T[name] = (np.ascontiguousarray(v, dtype=np.float32).view(np.uint32) >> 16).astype(np.uint16).reshape(shape)
    toks = [int(t) for t in rng.integers(0, V, 520)]
    steps = [[(0, 17)], [(0, 15), (1, 33)], [(0, 1), (1, 31), (2, 65)], [(0, 63), (2, 300)], [(1, 1), (2, 16), (0, 1)], [(2, 100)], [(0, 1), (1, 1), (2, 1)]]
    out = {}
    for dtype in ("float32", "bfloat16"):
        eng = q.Engine(spec, max_ctx=576, dtype=dtype).load_tensors(T)
        b, at, got = eng.batch(3, 576, page_tokens=page), [0, 0, 0], []
        for entries in steps:
            got.append(b.step([(m, toks[at[m]:at[m] + n]) for m, n in entries], range(sum(n for _, n in entries))))
            for m, n in entries:
                at[m] += n
        out[dtype] = np.concatenate(got)
        b.close()
        eng.close()
    want, got = out["float32"], out["bfloat16"]
    # a bf16 rounding is 2^-9 / sqrt(3) = 1.1e-3 of a value on the average, some ten of them stand one behind the other up to a logit: 3.6e-3 of
    # all rows, and half as much again for scores that a cap of 5 takes up to its slope.  A row of one wrong block would be 1e-1 and more.
    err = np.sqrt(((got - want) ** 2).mean(axis=1)) / want.std()
    assert np.isfinite(got).all() and np.sqrt((err ** 2).mean()) < 6e-3 and err.max() < 3e-2
