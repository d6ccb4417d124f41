"""Steps of 2 to 16 rows of layered bf16 engines, whose gate and up product has the activation in its epilogue (k_decode_bf16.hip kEpiGated),
against the float64 restatements: every activation; beside the mixer's rows in one product and alone; gate rows that are no whole tiles, mixer
rows that are none; rows of X in LDS and through the ring (width 5,248).  Held to the bf16 engines' tolerance."""
import numpy as np
import pytest

import test_gpu_layered as tivazen
import test_gpu_nukizen as nukizen
import test_gpu_sefelorn as sefelorn
import test_gpu_verelorn as verelorn
from nukizen_oracle import att, dense, lru, par

pytestmark = pytest.mark.gpu

MODELS = {
    "relu beside the mixer": (nukizen, [lru(width=30, mlp=dense(24)), att(mlp=dense(1000)), par(mlp=dense(8))], 640),
    "relu, wide": (nukizen, [att(mlp=dense(24)), lru(width=30, mlp=dense(40))], 5248),
    "clamped": (sefelorn, sefelorn.MIXED, 640),
    "gelu": (verelorn, verelorn.MIXED, 640),
    "silu": (tivazen, [tivazen.att(mlp=("dense", 40)), tivazen.att(mlp=("dense", 1000))], 640),
}


@pytest.mark.parametrize("name", MODELS)
def test_few_rows(name):
    mod, layers, width = MODELS[name]
    m = mod.Model(layers, seed=17, dtype="bfloat16", width=width)
    try:
        toks = m.tokens(60)
        want = m.ref(toks)
        got = mod.feed(m, 0, toks, [2, 16, 9, 3, 8, 15, 5, 2])
        d = np.sqrt(((got - want) ** 2).mean(axis=-1)) / np.std(want)
        assert max(np.quantile(d, 0.9), d.max() / 4) < m.tol
        # four slots' rows in one step
        for i in range(1, 4):
            m.batch.step([(i, toks[:20])], [19])
        at = m.batch.step([(i, toks[20:20 + n]) for i, n in ((1, 4), (2, 1), (3, 3))], range(8))
        ref = np.concatenate([want[20:24], want[20:21], want[20:23]])
        d = np.sqrt(((at - ref) ** 2).mean(axis=-1)) / np.std(want)
        assert max(np.quantile(d, 0.9), d.max() / 4) < m.tol
    finally:
        m.close()
