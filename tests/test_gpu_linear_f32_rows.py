"""fp32 products of the layered models in tiles of 32 rows (k_linear_f32.hip, lf::tile_rows): rows about the tiles' edges and the two limits of the rule,
experts of few rows and of none, against the numpy restatement; a row's bits beside as many others as take tiles of 64."""
import numpy as np
import pytest

from lugipel_oracle import attn, dense, moe
from test_gpu_lugipel import feed, model, rel  # noqa: F401

pytestmark = pytest.mark.gpu

TOL = 5e-5   # of the logits' spread: fp32 sums of up to 2,816 terms over three layers
LAYERS = [attn(heads=4, kv_heads=2, dim=64, vdim=64, size=70, mlp=dense(2816)),
          attn(heads=4, kv_heads=2, dim=64, vdim=64, size=70, mlp=moe(experts=8, identity=2, top=2, ff=352))]


@pytest.mark.parametrize("rows", [17, 31, 33, 64, 97, 128, 129, 224, 225, 480])
def test_rows(model, rows):  # noqa: F811
    m = model(LAYERS, seed=13, vocab=1003, width=256, slots=2, max_ctx=512)
    toks = m.tokens(rows)
    want = m.ref(toks)
    got = m.batch.step([(0, toks)], range(rows))
    assert rel(got, want) < TOL
    t = m.tokens(500 - rows if rows < 480 else 500)
    both = m.batch.step([(1, t)], range(len(t)))
    m.batch.release(0)
    m.batch.release(1)
    beside = m.batch.step([(1, t), (0, toks)], range(len(t) + rows))
    assert np.array_equal(beside[len(t):], got) and np.array_equal(beside[:len(t)], both)
