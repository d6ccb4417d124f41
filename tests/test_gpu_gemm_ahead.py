"""Products in two launches, whole rounds of 256x256 tiles for the first columns and smaller tiles for the rest (gemm_plan.hpp columns_ahead): every
epilogue, ragged columns, odd row strides, against fp32 products; and the rule itself on the host."""
import os
import random
import subprocess

import numpy as np
import pytest

import gpu_util as G
from gemm_route import CSRC
from qwen_inference_engine_amd import _lib
from test_gpu_gemm_mid import bf16, linear, products

DRIVER = r"""
#include "gemm_plan.hpp"
#include <cstdio>
int main() {
    long M, cols, K, cus;
    while (std::scanf("%ld %ld %ld %ld", &M, &cols, &K, &cus) == 4) std::printf("%ld\n", (long)qie::mid::columns_ahead(M, cols, K, cus, false));
}
"""
SHAPES = [(1030, 13500, 768), (700, 22004, 512), (511, 33001, 256), (2300, 7510, 256), (345, 45029, 768)]


def ahead(tmp_path, cases):
    (tmp_path / "d.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "d.cpp"), "-o", str(tmp_path / "d")], check=True)
    text = "\n".join("%d %d %d %d" % c for c in cases)
    return [int(v) for v in subprocess.run([str(tmp_path / "d")], input=text, text=True, capture_output=True, check=True).stdout.split()]


def test_the_rule_is_sound(tmp_path):
    """What goes ahead is whole column tiles in whole rounds of the chip, and something is left."""
    assert all(0 < a < N for (_, N, _), a in zip(SHAPES, ahead(tmp_path, [(*s, 256) for s in SHAPES])))
    r = random.Random(4)
    cases = [(r.randint(1, 9000), r.randint(8, 60000), 64 * r.randint(1, 300), r.choice([256, 304, 64])) for _ in range(3000)]
    got = ahead(tmp_path, cases)
    assert sum(a > 0 for a in got) > 100
    for (M, cols, K, cus), a in zip(cases, got):
        tiles = -(-M // 256) * (a // 256)
        assert a == 0 or (a % 256 == 0 and a < cols and M >= 256 and K >= 256 and (tiles % cus == 0 or cus - tiles % cus < -(-M // 256))), (M, cols, K, cus, a)


def test_a_rest_of_tall_tiles_and_long_k_stays(tmp_path):
    """Measured slower in two launches (748 against 770 and 781 us, 615 against 618)."""
    assert ahead(tmp_path, [(4880, 5120, 17408, 256), (5107, 5120, 17408, 256), (5120, 5120, 17408, 256), (6144, 4096, 14336, 256)]) == [0, 0, 0, 0]


PRICES = r"""
#include "gemm_plan.hpp"
#include <cstdio>
using namespace qie;
int main() {
    long M, cols, K, cus;
    while (std::scanf("%ld %ld %ld %ld", &M, &cols, &K, &cus) == 4) {
        const long a = (long)mid::columns_ahead(M, cols, K, cus, false), tiles = (M + 255) / 256 * (a / 256);
        const float more = M > mid::FITTED_ROWS ? 1.f : 1.06f;
        const float first = (tiles + cus - 1) / cus * (K / 64 * 1.45f + 5.f) + 5.f;   // unsplit
        const float one = std::min(g8p::us(M, cols, K, cus), more * mid::best(M, cols, K, cus).us);
        std::printf("%ld %.6g\n", a, a > 0 ? (first + more * mid::best(M, cols - a, K, cus).us) / one : 0.f);
    }
}
"""


def test_the_first_launch_is_priced_as_it_runs(tmp_path):
    """Never split over K, also where its tiles are fewer than the CUs (many row tiles: a round of the chip is few columns)."""
    r = random.Random(5)
    cases = [(23808, 1024, 18944, 256), (23571, 622, 19648, 256)] + [(r.randint(256, 32000), r.randint(300, 9000), 64 * r.randint(8, 330), 256) for _ in range(2000)]
    (tmp_path / "p.cpp").write_text(PRICES)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "p.cpp"), "-o", str(tmp_path / "p")], check=True)
    text = "\n".join("%d %d %d %d" % c for c in cases)
    got = [line.split() for line in subprocess.run([str(tmp_path / "p")], input=text, text=True, capture_output=True, check=True).stdout.splitlines()]
    assert sum(int(a) > 0 for a, _ in got) > 100
    for c, (a, of_one) in zip(cases, got):
        assert float(of_one) <= .9701, (c, a, of_one)


@pytest.mark.gpu
@pytest.mark.parametrize("M,rows,K", SHAPES)
@pytest.mark.parametrize("epi", ["f32", "store", "residual", "swiglu"])
def test_two_launches(qlib, oracle, M, rows, K, epi):
    N = rows // 2 if epi == "swiglu" else rows
    ld = N + 3
    x = bf16((M, K), 1.0, 21)
    if epi == "swiglu":
        wg, wu, y0 = bf16((N, K), 1.5 * K ** -0.5, 22), bf16((N, K), K ** -0.5, 23), bf16((M + 1, ld), 1.0, 24)
        y = G.dev(y0)
        linear(G.dev(x), [G.dev(wg), G.dev(wu)], [], M, K, N, y, _lib.QIE_EPI_SWIGLU, ldy=ld)
        (g, gs), (u, us) = products(x, wg), products(x, wu)
        want = u / (1.0 + np.exp(-g)) * g
        # |silu'| <= 1.1; three bf16 roundings (gate, silu, product) and one of the up sum
        tol = 2.0 ** -7 * (np.abs(want) + 1.1 * np.abs(u) * np.abs(g)) + 1e-5 * (1.1 * np.abs(u) * gs + np.abs(g) * us)
    else:
        w = bf16((N, K), K ** -0.5, 22)
        acc, scale = products(x, w)
        if epi == "f32":
            y = G.zeros((M, N), np.float32)
            linear(G.dev(x), [G.dev(w)], [], M, K, N, y, _lib.QIE_EPI_F32)
            assert (np.abs(y.numpy() - acc) <= 1e-5 * scale).all()
            return
        y0 = bf16((M + 1, ld), 1.0, 24)
        y = G.dev(y0)
        if epi == "store":
            b = bf16((N,), 0.5, 25)
            linear(G.dev(x), [G.dev(w)], [G.dev(b)], M, K, N, y, _lib.QIE_EPI_STORE, ldy=ld)
            want = acc + G.bf(b)
            tol = 2.0 ** -8 * np.abs(want) + 1e-5 * scale
        else:
            linear(G.dev(x), [G.dev(w)], [], M, K, N, y, _lib.QIE_EPI_RESIDUAL, ldy=ld)
            want = G.bf(y0)[:M, :N] + G.bf(oracle.f32_to_bf16(acc))
            # bf16(res + bf16(acc)): an ulp of either rounding
            tol = 2.0 ** -7 * (np.abs(acc) + np.abs(want)) + 1e-5 * scale
    got = G.host_bf16(y)
    assert (np.abs(G.bf(got)[:M, :N] - want) <= tol).all()
    assert np.array_equal(got[:M, N:], y0[:M, N:]) and np.array_equal(got[M], y0[M])


@pytest.mark.gpu
def test_fp32_results_keep_their_error(qlib):
    """Of a product whose columns would go ahead with bf16 results.  An fp32 chain's error grows with the square root of its steps, so one chain over K errs
    by sqrt(2) of what two over halves of it do: 1.55e-7 and 1.10e-7 of the result here, over 14 million of them.  The bound is their geometric mean."""
    M, N, K = 1030, 13500, 768
    x, w = bf16((M, K), 1.0, 41), bf16((N, K), K ** -0.5, 42)
    y = G.zeros((M, N), np.float32)
    linear(G.dev(x), [G.dev(w)], [], M, K, N, y, _lib.QIE_EPI_F32)
    want = G.bf(x).astype(np.float64) @ G.bf(w).astype(np.float64).T
    err = np.linalg.norm(y.numpy() - want) / np.linalg.norm(want)
    assert err <= 1.31e-7, err
