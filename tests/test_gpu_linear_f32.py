"""fp32 products of the layered models on the matrix cores at the sizes where they can go wrong: 1 to 16 rows (k_decode_bf16.hip's
fp32 form: X in LDS and through the ring), 17 to 300 (k_linear_f32.hip: whole and split tiles, ragged rows and columns, experts of
few and of no rows), widths off their grid (the plain kernels); and the exact attention at head sizes on and off four elements."""
import ctypes as C

import numpy as np
import pytest

import gpu_util as G
from lugipel_oracle import attn, dense, gru, moe
from qwen_inference_engine_amd import _lib
from test_gpu_gemm_mid import GROWS
from test_gpu_lugipel import feed, model, rel  # noqa: F401  (model: a fixture)

pytestmark = pytest.mark.gpu

TOL = 5e-5   # of the logits' spread: fp32 sums of up to 2,816 terms over three layers

LAYERS = {
    "dense": [attn(heads=4, kv_heads=2, dim=64, vdim=64, size=70, mlp=dense(2816)), gru(width=320, mlp=dense(96))],
    "routed": [gru(width=256, mlp=moe(experts=7, identity=1, top=2, count=2, keep=1, ff=64)), attn(heads=4, kv_heads=1, dim=32, vdim=96, size=300, mlp=None)],
    "odd heads": [attn(heads=3, kv_heads=3, dim=30, vdim=65, size=33, mlp=dense(72)), attn(heads=2, kv_heads=1, dim=130, vdim=257, size=9, mlp=None)],
}


@pytest.mark.parametrize("width", [256, 272])   # 272: off the 64 grid, on the 16 grid
@pytest.mark.parametrize("layers", sorted(LAYERS))
def test_rows(model, layers, width):  # noqa: F811
    m = model(LAYERS[layers], seed=7, vocab=1003, width=width, slots=6, max_ctx=512)
    toks = m.tokens(302)
    want = m.ref(toks)
    sizes = [1, 2, 8, 9, 15, 16, 17, 33, 64, 65, 72]      # 302 rows in all
    assert sum(sizes) == 302 and rel(feed(m, 0, toks, sizes), want) < TOL
    assert rel(feed(m, 1, toks, [302]), want) < TOL
    # sixteen rows as single tokens and short portions of several slots
    a, b = [m.tokens(5) for _ in range(4)], m.tokens(12)
    out = m.batch.step([(2 + i, t[:1]) for i, t in enumerate(a)] + [(0, b)], range(16))
    for i, t in enumerate(a):
        assert rel(out[i:i + 1], m.ref(t[:1])) < TOL
    assert rel(out[4:], m.ref(toks + b)[302:]) < TOL


def test_replay_after_larger_steps(model):  # noqa: F811
    """Captured steps keep their split-K memory: steps of 16 rows with four experts each replay after larger steps, a prompt of another
    batch on the same engine, and a product on its stream that outgrows the memory the capture has seen."""
    layers = [gru(width=256, mlp=moe(experts=8, identity=0, top=4, count=1, keep=1, ff=256)), attn(heads=4, kv_heads=2, dim=64, vdim=64, size=40, mlp=None)]
    m = model(layers, seed=3, vocab=1003, width=256, slots=4, max_ctx=512)
    seqs = [[], []]

    def small():
        t = [m.tokens(8), m.tokens(8)]
        out = m.batch.step([(0, t[0]), (1, t[1])], range(16))
        for i in range(2):
            seqs[i] += t[i]
            assert rel(out[8 * i:8 * i + 8], m.ref(seqs[i])[-8:]) < TOL
    for _ in range(8):
        small()
    graphs, before = m.batch.graph_stats()
    assert graphs > 0 and before > 0
    for n in (60, 64):
        t = m.tokens(n)
        assert rel(m.batch.step([(2, t)], range(n)), m.ref(t)) < TOL
        m.batch.release(2)
        for _ in range(3):
            small()
    other = m.eng.batch(1, 512, page_tokens=16)
    t = m.tokens(300)
    assert rel(other.step([(0, t)], range(300)), m.ref(t)) < TOL
    for _ in range(3):
        small()
    other.close()
    M, N, K = GROWS
    a, x, w, y = _lib.LinearArgsC(), G.zeros_bf16(M, K), G.zeros_bf16(N, K), G.dev(np.full((M, N), 7.0, np.float32))
    a.x, a.ldx, a.w[0], a.seg_rows[0], a.M, a.K, a.N, a.y, a.ldy, a.epilogue = G.p(x), K, G.p(w), N, M, K, N, G.p(y), N, _lib.QIE_EPI_F32
    for _ in range(2):
        G.check(_lib.load().qie_linear(C.byref(a), m.eng.stream), "qie_linear")
        for _ in range(3):
            small()
    assert not y.numpy().any()
    assert m.batch.graph_stats()[1] > before + 12


@pytest.mark.parametrize("width", [2048, 3072])   # X in LDS, through the ring
def test_sums_of_equal_terms(model, width):  # noqa: F811
    """Few rows, every product of a sum the same: a serial chain of fp32 additions drifts off by up to half an ulp of the running
    sum each (width / 8 terms: 60 to 90 units of 2^-24), sums of width / 128 terms that meet in pairs cannot."""
    def tweak(T, cfg):
        T["l0.mix.o"][:] = 0                                             # the row stays what the embedding makes it
        T["embed"][:] = np.where(np.arange(width) % 2 == 0, 2.0, 0.0)    # with position 0's sines and cosines: ones
        T["final.norm"][:] = 1.0
        T["head"][:] = (1.0 + np.arange(8) / 64.0)[np.arange(503) % 8, None]
    m = model([gru(width=64, mlp=None)], seed=5, vocab=503, width=width, slots=16, max_ctx=64, tweak=tweak)
    want = width * m.W64["head"][:, 0] / np.sqrt(1.0 + 1e-5)
    # a chain's terms and the seven pairings of 16 x 8 sums, a rounding each; four more for the norm's quotient, its root and its products
    bound = (width // 128 + 7 + 4) * 2.0 ** -24
    for rows in (1, 5, 16):
        got = m.batch.step([(i, m.tokens(1)) for i in range(rows)], range(rows))
        assert (np.abs(got / want - 1.0) <= bound).all()
        for i in range(rows):
            m.batch.release(i)


def test_rows_beside_others(model):  # noqa: F811
    """A prompt's logits are the same bits alone and beside other prompts (more rows: fewer workgroups share a tile's sums)."""
    layers = [attn(heads=4, kv_heads=2, dim=64, vdim=64, size=70, mlp=dense(1440)), attn(heads=4, kv_heads=2, dim=64, vdim=64, size=70, mlp=moe(experts=6, identity=2, top=2, ff=352))]
    m = model(layers, seed=9, vocab=1003, width=512, slots=3, max_ctx=512)
    t, others = m.tokens(40), [m.tokens(30), m.tokens(400)]
    want = m.batch.step([(0, t)], range(40))
    assert rel(want, m.ref(t)) < TOL
    for o in others:
        m.batch.release(0)
        m.batch.release(1)
        assert np.array_equal(m.batch.step([(1, o), (0, t)], range(len(o), len(o) + 40)), want)
        m.batch.release(0)
        m.batch.release(1)
        assert np.array_equal(m.batch.step([(0, t), (1, o)], range(40 + len(o)))[:40], want)
