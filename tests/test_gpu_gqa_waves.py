"""The layered attention on exact rows (k_mixers.hip): blocks of 16 waves beside those of 4, against the numpy restatement."""
import pytest

from lugipel_oracle import attn
from test_gpu_lugipel import feed, model, rel  # noqa: F401

pytestmark = pytest.mark.gpu


def test_attention_in_blocks_of_either_size(model):  # noqa: F811
    """Steps of 85 rows and fewer (6 heads) take 16 waves a block, longer ones 4; contexts of one chunk of 256 keys and of two."""
    m = model([attn(heads=6, kv_heads=3, dim=6, vdim=10, size=400), attn(heads=6, kv_heads=2, dim=8, vdim=70, size=300)], seed=3)
    toks = m.tokens(420)
    want = m.ref(toks)
    got = feed(m, 0, toks, [85, 86, 100, 60, 3, 1, 85])
    assert rel(got, want) < m.tol
