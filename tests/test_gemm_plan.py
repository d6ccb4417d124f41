"""CPU: the plans of the split GEMMs (csrc/gemm_plan.hpp), compiled with the host compiler."""
import os
import random
import subprocess

import pytest

from test_gpu_gemm_mid import GROWS, PLANS

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen_inference_engine_amd", "csrc")

DRIVER = r"""
#include "gemm_plan.hpp"
#include <cstdio>
#include <vector>
// "m M columns K cus": plan of k_gemm_mid.hip; "f M N K batch grouped cus": k_linear_f32.hip; "t M N K groups off[0] .. off[groups]": its row tiles' indices
int main() {
    char op;
    while (std::scanf(" %c", &op) == 1) {
        long M, N, K, batch, x, cus;
        if (op == 'm') {
            if (std::scanf("%ld %ld %ld %ld", &M, &N, &K, &cus) != 4) return 2;
            const qie::mid::Plan p = qie::mid::plan(M, N, K, cus);
            std::printf("%d %d %d %d\n", p.tile, p.whole, p.splitk, p.n_mt * p.n_nt);
        } else if (op == 'f') {
            if (std::scanf("%ld %ld %ld %ld %ld %ld", &M, &N, &K, &batch, &x, &cus) != 6) return 2;
            const qie::lf::Plan p = qie::lf::plan(M, N, K, batch, x != 0, cus);
            std::printf("%d %d %d %d %ld\n", p.n_nt, p.n_mt, p.log_segs, p.log_parts, (long)p.row_tiles);
        } else {
            if (std::scanf("%ld %ld %ld %ld", &M, &N, &K, &batch) != 4) return 2;
            std::vector<int> off(batch + 1);
            for (int& o : off)
                if (std::scanf("%d", &o) != 1) return 2;
            const qie::lf::Plan p = qie::lf::plan(M, N, K, batch, true, 256);
            for (int z = 0; z < batch; z++)   // the grid, as the kernel walks it
                for (int mt = 0; mt < p.n_mt; mt++) {
                    const int m0 = off[z] + mt * qie::lf::BM;
                    if (m0 < off[z + 1]) std::printf("%ld ", (long)qie::lf::row_tile(true, m0, z, mt, p.n_mt));
                }
            std::printf("\n");
        }
    }
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "drive.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(d / "drive.cpp"), "-o", str(d / "drive")], check=True)

    def run(lines):
        out = subprocess.run([str(d / "drive")], input="\n".join(lines), text=True, capture_output=True, check=True).stdout
        return [[int(v) for v in line.split()] for line in out.splitlines()]
    return run


def test_gemm_mid_shapes_take_every_tile(plan):
    """The shapes that the GPU test multiplies have the plans it says, every tile among them whole, split and both."""
    got = [(p[0], "whole" if p[2] == 1 else "split" if p[1] == 0 else "mixed") for p in plan([f"m {M} {N} {K} 256" for M, N, K, _, _ in PLANS])]
    assert got == [(t, kind) for _, _, _, t, kind in PLANS]
    assert set(got) == {(t, kind) for t in range(8) for kind in ("whole", "split", "mixed")}


def test_a_shape_whose_slabs_outgrow_the_reserve(plan):
    (tile, whole, splitk, tiles), = plan(["m %d %d %d 256" % GROWS])
    bm, bn = [(64, 64), (64, 128), (128, 64), (128, 128), (192, 128), (256, 128), (320, 64), (320, 128)][tile]
    assert splitk > 1 and (tiles - whole) * splitk * bm * bn * 4 > 64 << 20


def test_gemm_mid_plans_are_sound(plan):
    """Whole tiles are whole rounds of the chip or all of them, and a split leaves every part a k-tile."""
    r = random.Random(3)
    cases = [(int(2 ** r.uniform(4.1, 13)), int(2 ** r.uniform(3, 18)), 64 * int(2 ** r.uniform(0, 9)), r.choice([256, 256, 304, 64])) for _ in range(3000)]
    for (M, N, K, cus), (tile, whole, splitk, tiles) in zip(cases, plan(["m %d %d %d %d" % c for c in cases])):
        assert tile in range(8) and 1 <= splitk <= min(12, K // 64) and 0 <= whole <= tiles
        assert whole == tiles if splitk == 1 else whole < tiles and whole % cus == 0


@pytest.mark.parametrize("seed", range(6))
def test_row_tiles_of_groups(plan, seed):
    """Every row tile of every group has an index of its own, below the plan's count."""
    r = random.Random(seed)
    for _ in range(20):
        groups, M = r.randint(1, 40), r.randint(33, 1500)
        total = r.randint(0, M)   # the rest are rows that no group owns
        cuts = sorted(r.choice([0, total, r.randint(0, total)]) for _ in range(groups - 1))
        off = [0] + cuts + [total]
        tiles, p = plan([f"t {M} 1024 1024 {groups} " + " ".join(map(str, off)), f"f {M} 1024 1024 {groups} 1 256"])
        assert len(set(tiles)) == len(tiles) and all(0 <= t < p[4] for t in tiles)


def test_slabs_are_bounded(plan):
    """Partial tiles take the memory of the tiles that exist: 32 MB at most on 256 CUs (1,024 parts of 32 KB)."""
    r = random.Random(7)
    cases = [(int(2 ** r.uniform(4.1, 13)), int(2 ** r.uniform(4, 15)), 32 * int(2 ** r.uniform(0, 9)), r.choice([1, 1, 2, 8, 16, 64, 128]), r.randint(0, 1)) for _ in range(400)]
    cases += [(2048, 256, 1024, 8, 1), (240, 1408, 1024, 8, 1), (240, 1024, 704, 8, 1)]
    for c, (n_nt, n_mt, segs, parts, row_tiles) in zip(cases, plan([f"f {' '.join(map(str, c))} 256" for c in cases])):
        assert 0 <= parts <= segs <= 4
        assert segs == 0 or c[2] // 32 >> segs >= 8      # a segment keeps eight k-tiles
        if parts:
            assert (row_tiles * n_nt << parts) * 8192 * 4 <= 32 << 20


def test_segments_follow_k_alone(plan):
    for K in (32, 96, 256, 1024, 1056, 2816, 16384):
        got = {p[2] for p in plan([f"f {M} {N} {K} {b} {g} {cus}" for M in (17, 64, 300, 4000) for N in (64, 1000, 32000) for b, g in ((1, 0), (8, 0), (8, 1)) for cus in (256, 304)])}
        assert len(got) == 1
