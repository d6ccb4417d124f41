"""The layered attention on exact rows (k_mixers.hip): blocks of 16 waves beside those of 4, against the numpy restatement."""
import numpy as np
import pytest

from lugipel_oracle import attn, dense
from test_gpu_lugipel import feed, model, rel  # noqa: F401

pytestmark = pytest.mark.gpu


def test_attention_in_blocks_of_either_size(model):  # noqa: F811
    """Steps of 85 rows and fewer (6 heads) take 16 waves a block, longer ones 4; contexts of one chunk of 256 keys and of two."""
    m = model([attn(heads=6, kv_heads=3, dim=6, vdim=10, size=400), attn(heads=6, kv_heads=2, dim=8, vdim=70, size=300)], seed=3)
    toks = m.tokens(420)
    want = m.ref(toks)
    got = feed(m, 0, toks, [85, 86, 100, 60, 3, 1, 85])
    assert rel(got, want) < m.tol


def test_bits_do_not_depend_on_the_blocks(model):  # noqa: F811
    """Rows of more than 16 in a step, so that the products' kernels are the same: steps of either kind, one chunk of keys and two."""
    m = model([attn(heads=6, kv_heads=3, dim=64, vdim=64, size=400, mlp=dense(1440)), attn(heads=6, kv_heads=2, dim=64, vdim=128, size=300, mlp=dense(1440))],
              seed=4, width=512, vocab=503)
    toks = m.tokens(420)
    whole = m.batch.step([(0, toks)], range(420))
    m.batch.release(0)
    assert np.array_equal(feed(m, 0, toks, [85, 86, 100, 64, 85]), whole)
