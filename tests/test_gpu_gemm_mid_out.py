"""What every tile of k_gemm_mid.hip writes: its residual and SwiGLU epilogues, whole and split over K, by quads and by elements, against fp32
products; nothing behind a row's columns or behind the last row.  128, 192 and 256 x 128 in both of their forms (parts of K below and from
4,096, over many row tiles 2,304, 1,280 and 1,792; one row tile: 6,144)."""
import numpy as np
import pytest

import gpu_util as G
from gemm_route import routes
from qwen_inference_engine_amd import _lib
from test_gpu_gemm_mid import bf16, linear, products

pytestmark = pytest.mark.gpu

# rows, weight rows, K, tile, parts (gate and up of up to 32 rows: k_gemm_few.hip)
SHAPES = [(17, 72, 64, 0, 1), (35, 104, 128, 0, 1), (33, 72, 12416, 0, 9), (17, 16500, 64, 1, 1), (35, 112, 192, 1, 1), (64, 8200, 4096, 1, 3), (65, 8200, 1024, 2, 1), (129, 4000, 4096, 2, 2),
          (301, 9728, 896, 3, 1), (128, 8200, 4096, 3, 3), (131, 11014, 3712, 4, 2), (210, 9278, 6464, 5, 3), (640, 4000, 4096, 6, 2),
          (257, 8338, 11264, 7, 3), (127, 16500, 64, 8, 1), (640, 8200, 448, 9, 1), (395, 10424, 256, 4, 1), (276, 15640, 1152, 4, 1),
          (439, 15744, 512, 5, 1), (213, 22912, 1536, 5, 1), (216, 12496, 5120, 3, 1), (467, 3512, 8192, 3, 2),
          (104, 16500, 2048, 3, 1), (649, 7496, 1536, 4, 1), (1008, 7600, 2048, 5, 1), (393, 4688, 3072, 4, 2),
          (469, 7088, 8192, 5, 2)]


def test_the_shapes_take_their_tiles():
    for gated in (0, 1):
        got = [(r["tile"], r["splitk"], r["ahead"]) for r in routes([(*s[:3], gated, 0) for s in SHAPES])]
        assert got == [(-2 if gated and s[0] <= 32 else s[3], s[4], 0) for s in SHAPES]


@pytest.mark.parametrize("M,rows,K,tile,parts", SHAPES)
@pytest.mark.parametrize("odd", [0, 1])
@pytest.mark.parametrize("epi", ["residual", "swiglu"])
def test_writes_its_part_of_the_rows(qlib, oracle, M, rows, K, tile, parts, odd, epi):
    N = rows // 2 if epi == "swiglu" else rows
    N -= odd                      # odd: element by element
    ld = N + (4 if not odd else 3)
    x, y0 = bf16((M, K), 1.0, 11), bf16((M + 1, ld), 1.0, 12)
    y = G.dev(y0)
    if epi == "residual":
        w = bf16((N, K), K ** -0.5, 13)
        linear(G.dev(x), [G.dev(w)], [], M, K, N, y, _lib.QIE_EPI_RESIDUAL, ldy=ld)
        acc, scale = products(x, w)
        want = G.bf(y0)[:M, :N] + G.bf(oracle.f32_to_bf16(acc))
        # bf16(res + bf16(acc)): an ulp of either rounding
        tol = 2.0 ** -7 * (np.abs(acc) + np.abs(want)) + 1e-5 * scale
    else:
        wg, wu = bf16((N, K), 1.5 * K ** -0.5, 14), bf16((N, K), K ** -0.5, 15)
        linear(G.dev(x), [G.dev(wg), G.dev(wu)], [], M, K, N, y, _lib.QIE_EPI_SWIGLU, ldy=ld)
        (g, gs), (u, us) = products(x, wg), products(x, wu)
        want = u / (1.0 + np.exp(-g)) * g
        # |silu'| <= 1.1; three bf16 roundings (gate, silu, product) and one of the up sum
        tol = 2.0 ** -7 * (np.abs(want) + 1.1 * np.abs(u) * np.abs(g)) + 1e-5 * (1.1 * np.abs(u) * gs + np.abs(g) * us)
    got = G.host_bf16(y)
    assert (np.abs(G.bf(got)[:M, :N] - want) <= tol).all()
    assert np.array_equal(got[:M, N:], y0[:M, N:]) and np.array_equal(got[M], y0[M])
