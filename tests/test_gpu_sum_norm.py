"""A prompt's projection with its residual and the norm behind it (gemm_add_norm), where K is cut into parts that the norm's launch adds up: both of
k_gemm_few.hip's and k_gemm_mid.hip's tiles, ragged rows, one part and many, both norms' numerics, every number of 2,048-column vectors a row, and shapes
that stay two launches."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import gpu_util as G
from qwen_inference_engine_amd import _lib
from test_gpu_gemm_mid import bf16, products

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen_inference_engine_amd", "csrc")
SYMBOL = "_ZN3qie13gemm_add_normEPK15qie_linear_argsPKvfiPvP12ihipStream_t"
DRIVER = r"""
#include "gemm_plan.hpp"
#include <cstdio>
int main() {
    long M, N, K;
    while (std::scanf("%ld %ld %ld", &M, &N, &K) == 3) {
        const qie::apart::Plan p = qie::apart::choose(M, N, K, 256);
        std::printf("%d %d %d\n", p.form, p.tile, p.parts);
    }
}
"""
# rows, columns, K
SHAPES = [(17, 896, 896), (24, 896, 4864), (33, 904, 4864), (113, 896, 4864), (113, 3584, 3584), (113, 3584, 18944), (200, 1536, 8960), (301, 3584, 18944),
          (301, 5120, 5120), (257, 896, 896), (257, 7168, 2048), (800, 896, 4864), (129, 16, 1024), (640, 3584, 18944), (24, 5120, 17408), (257, 5120, 5120), (512, 896, 4864)]
APART_NOT = [(16, 896, 4864), (113, 896, 4872), (1100, 3584, 3584), (300, 8448, 1024)]   # few rows, K off the grid of 64, many rows, rows of more than 8,192


def plans(tmp_path, cases):
    (tmp_path / "drive.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "drive.cpp"), "-o", str(tmp_path / "drive")], check=True)
    out = subprocess.run([str(tmp_path / "drive")], input="\n".join("%d %d %d" % c for c in cases), text=True, capture_output=True, check=True).stdout
    return [tuple(int(v) for v in line.split()) for line in out.splitlines()]


def test_plans(tmp_path):
    """The shapes below come in forms and tiles, one part and many; every plan's parts have work and fit what a stream holds from the start."""
    got = plans(tmp_path, SHAPES)
    assert all(f >= 0 or t >= 0 for f, t, _ in got)
    assert {f for f, _, _ in got} >= {-1, 0, 1, 2, 3} and len({t for _, t, _ in got}) >= 5 and {p for _, _, p in got} >= {1, 2, 9}, got
    assert plans(tmp_path, APART_NOT[:3]) == [(-1, -1, 1)] * 3
    r = np.random.default_rng(1)
    cases = [(int(2 ** r.uniform(4, 11)), 8 * int(2 ** r.uniform(1, 10)), 64 * int(2 ** r.uniform(0, 9))) for _ in range(2000)]
    for (M, N, K), (f, t, p) in zip(cases, plans(tmp_path, cases)):
        assert (f >= 0) + (t >= 0) <= 1 and 1 <= p <= max(1, min(16, K // 64)) and p * M * N <= (16 << 20 if p > 1 else 1 << 40)


# rows, columns, K, us apart and in the parts that the fit prefers or has on a level
MEASURED = [(400, 1024, 2816, 11.2, 12.7), (640, 2048, 2048, 20.5, 22.1), (301, 2048, 2048, 13.5, 14.8), (512, 1024, 1024, 8.2, 9.0), (512, 512, 1536, 7.8, 8.4),
            (301, 512, 2048, 7.8, 8.8), (17, 3584, 18944, 30.6, 27.1), (113, 5120, 17408, 55.1, 46.0), (80, 5120, 5120, 23.4, 22.0), (113, 896, 896, 6.73, 6.57)]


def test_plans_that_measured_longer_are_not_taken(tmp_path):
    for c, (f, t, _) in zip(MEASURED, plans(tmp_path, [c[:3] for c in MEASURED])):
        assert (f >= 0 or t >= 0) == (c[4] < c[3]), c


@pytest.mark.gpu
@pytest.mark.parametrize("numerics", [_lib.QIE_NUMERICS_REF, _lib.QIE_NUMERICS_HF])
@pytest.mark.parametrize("M,N,K", SHAPES + APART_NOT[1:])
def test_as_product_and_norm(qlib, oracle, M, N, K, numerics):
    ldx = K + 8
    x, w, res, nw = bf16((M, ldx), 1.0, 1), bf16((N, K), K ** -0.5, 2), bf16((M, N), 1.0, 3), bf16((N,), 1.0, 4)
    dx, dw, dn = G.dev(x), G.dev(w), G.dev(nw)
    fn = getattr(C.CDLL(_lib.load()._name), SYMBOL)
    fn.restype, fn.argtypes = C.c_int, [C.c_void_p, C.c_void_p, C.c_float, C.c_int, C.c_void_p, C.c_void_p]
    out = []
    for _ in range(2):
        y, h = G.dev(res), G.zeros_bf16(M, N)
        a = _lib.LinearArgsC()
        a.x, a.ldx, a.M, a.K, a.N, a.y, a.ldy, a.epilogue = G.p(dx), ldx, M, K, N, G.p(y), N, _lib.QIE_EPI_RESIDUAL
        a.w[0], a.seg_rows[0] = G.p(dw), N
        G.check(fn(C.byref(a), G.p(dn), 1e-6, numerics, G.p(h), None), "gemm_add_norm")
        out.append((G.host_bf16(y), G.host_bf16(h)))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])   # parts in their order
    acc, scale = products(x[:, :K], w)
    want = G.bf(res) + G.bf(oracle.f32_to_bf16(acc))
    got = G.bf(out[0][0])
    # bf16(res + bf16(acc)): an ulp of either rounding
    assert (np.abs(got - want) <= 2.0 ** -7 * (np.abs(acc) + np.abs(want)) + 1e-5 * scale).all()
    # the norm is qie_rmsnorm's of the rows that were written, bit for bit
    z, h = G.dev(out[0][0]), G.zeros_bf16(M, N)
    G.check(qlib.qie_rmsnorm(G.p(z), G.p(dn), G.p(h), M, N, 1e-6, numerics, None), "qie_rmsnorm")
    assert np.array_equal(out[0][1], G.host_bf16(h))
