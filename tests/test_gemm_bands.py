"""CPU: the order in which the GEMMs' workgroups take their tiles (csrc/gemm_plan.hpp), compiled with the host compiler."""
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen_inference_engine_amd", "csrc")

DRIVER = r"""
#include "gemm_plan.hpp"
#include <cstdio>
// "n_mt n_nt bm bn at_once": the band height, then every workgroup's tile
int main() {
    int n_mt, n_nt, bm, bn, at_once;
    while (std::scanf("%d %d %d %d %d", &n_mt, &n_nt, &bm, &bn, &at_once) == 5) {
        const int gm = qie::band_height(n_mt, bm, bn, at_once);
        std::printf("%d", gm);
        for (int wid = 0; wid < n_mt * n_nt; wid++) {
            int mt, nt;
            qie::banded(wid, n_mt, n_nt, gm, &mt, &nt);
            std::printf(" %d", nt * n_mt + mt);
        }
        std::printf("\n");
    }
}
"""


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    d = tmp_path_factory.mktemp("bands")
    (d / "drive.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(d / "drive.cpp"), "-o", str(d / "drive")], check=True)

    def run(cases):
        text = "\n".join(" ".join(map(str, c)) for c in cases)
        out = subprocess.run([str(d / "drive")], input=text, text=True, capture_output=True, check=True).stdout
        return [[int(v) for v in line.split()] for line in out.splitlines()]
    return run


def test_bands_take_every_tile_once(order):
    r = random.Random(1)
    sizes = [(64, 64, 64), (64, 128, 64), (128, 64, 64), (320, 128, 32), (256, 256, 32)]
    cases = [(m, n) + s for m in (1, 2, 8, 9, 15, 16, 17, 33) for n in (1, 5, 14) for s in sizes]
    cases += [(r.randint(1, 80), r.randint(1, 40)) + r.choice(sizes) for _ in range(100)]
    for (n_mt, n_nt, _, _, _), (gm, *tiles) in zip(cases, order(cases)):
        assert 1 <= gm <= n_mt
        assert sorted(tiles) == list(range(n_mt * n_nt))
        if n_mt < 8:
            assert gm == n_mt or gm * 2 >= n_mt   # few row tiles: one band, or two
