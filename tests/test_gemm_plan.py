"""CPU: the plans of the split GEMMs (csrc/gemm_plan.hpp), compiled with the host compiler."""
import os
import random
import subprocess

import pytest

from gemm_route import routes
from test_gpu_gemm_mid import GROWS, MORE, PLANS, SHAPES

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen_inference_engine_amd", "csrc")

DRIVER = r"""
#include "gemm_plan.hpp"
#include <cstdio>
#include <vector>
// "m M columns K cus": plan of k_gemm_mid.hip; "s ldx ldy": whether it takes such rows; "f M N K batch grouped cus": k_linear_f32.hip; "t M N K groups off[0] .. off[groups]": its row tiles' indices
int main() {
    char op;
    while (std::scanf(" %c", &op) == 1) {
        long M, N, K, batch, x, cus;
        if (op == 'm') {
            if (std::scanf("%ld %ld %ld %ld", &M, &N, &K, &cus) != 4) return 2;
            const qie::mid::Plan p = qie::mid::plan(M, N, K, cus);
            std::printf("%d %d %d %d\n", p.tile, p.whole, p.splitk, p.n_mt * p.n_nt);
        } else if (op == 's') {
            if (std::scanf("%ld %ld", &M, &N) != 2) return 2;
            std::printf("%d\n", qie::mid::strides_fit(M, N) ? 1 : 0);
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


def test_gemm_mid_products_come_to_every_tile():
    """What qie_linear does with the shapes that the GPU test multiplies, one segment each: every tile whole, split and both, but for two that are mixed
    only where a tile of 160 columns is the better one."""
    got = {(r["tile"], "whole" if r["splitk"] == 1 else "split" if r["whole"] == 0 else "mixed") for r in routes(SHAPES + MORE, f32=True) if r["tile"] >= 0 and r["ahead"] == 0}
    assert {g for g in got if g[0] < 8} == {(t, kind) for t in range(8) for kind in ("whole", "split", "mixed")} - {(2, "mixed"), (6, "mixed")}
    (r,) = routes([GROWS], f32=True)
    assert 0 <= r["tile"] < 8 and r["splitk"] > 1 and r["ahead"] == 0


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


def test_gemm_mid_offsets_fit(plan):
    """Rows so far apart that a tile's offsets would wrap go to other kernels: 32 bits of bytes for x, 31 for y, of 4 bytes an element."""
    rows, cols = 320, 160   # of the tallest and the widest tile
    r = random.Random(6)
    strides = [int(2 ** r.uniform(6, 40)) for _ in range(2000)] + [1 << 20, (1 << 20) + 8, 1 << 22, (1 << 22) + 8, 6731912, 6731920, 6731928, 7158280]
    taken = [x for x, (t,) in zip(strides, plan([f"s {x} 64" for x in strides])) if t]
    assert max(taken) >= 1 << 22 and all(((rows - 1) * x + 64) * 2 < 1 << 32 for x in taken)
    taken = [y for y, (t,) in zip(strides, plan([f"s 64 {y}" for y in strides])) if t]
    assert max(taken) >= 1 << 20 and all((rows * y + cols) * 4 < 1 << 31 for y in taken)


# rows, weight rows, K, us as 128 x 64 tiles in two parts of K and as whole 64 x 64 tiles
SMALL = [(193, 3584, 3584, 18.1, 16.4), (220, 3584, 3584, 18.5, 17.5), (230, 3584, 3584, 18.8, 18.2), (245, 3584, 3584, 19.2, 19.7), (193, 2560, 2560, 13.8, 11.9),
         (230, 2560, 2560, 13.9, 12.1), (129, 5120, 5120, 25.7, 22.1), (166, 5120, 5120, 27.6, 27.3)]


def test_small_tiles_with_a_last_row_tile_hardly_filled():
    """The plan's choice between the two (at 245 rows k_gemm_few.hip takes the product before it is asked)."""
    for (M, N, K, split, whole), r in zip(SMALL, routes([c[:3] for c in SMALL])):
        assert (r["mid"], r["splitk"]) == ((0, 1) if whole < split else (2, 2)), (M, N, K, r)


# rows, weight rows, K, us of the best of the other tiles and the 256x256 kernel, of the 160-column tiles 8 to 11
MEASURED = [
    (400, 9728, 896, 18.1, [16.9, 21.1, 24.8, 29.8]),
    (1024, 9728, 896, 30.6, [30.8, 39.7, 26.3, 31.2]),
    (1600, 9728, 896, 47.5, [59.4, 57.1, 48.0, 57.4]),
    (3500, 9728, 896, 91.7, [105.2, 98.9, 96.7, 88.6]),
    (100, 37888, 3584, 69.7, [57.5, 62.8, 71.6, 81.8]),
    (300, 37888, 3584, 122.1, [122.3, 110.7, 129.8, 96.1]),
    (512, 37888, 3584, 168.9, [173.9, 164.5, 135.5, 161.9]),
    (640, 37888, 3584, 166.7, [215.4, 213.9, 193.0, 179.1]),
    (960, 37888, 3584, 252.5, [328.6, 272.9, 261.0, 260.7]),
    (640, 28672, 4096, 162.0, [192.0, 182.6, 213.0, 190.1]),
    (640, 34816, 5120, 225.3, [304.4, 295.5, 266.5, 245.4]),
    (4096, 4608, 3584, 159.1, [166.0, 156.0, 133.8, 155.4]),
    (8192, 4608, 3584, 249.0, [331.3, 266.4, 254.2, 240.3]),
    (6000, 3584, 3584, 175.5, [210.6, 168.2, 198.5, 167.5]),
    (7000, 7168, 5120, 448.3, [546.7, 495.9, 460.0, 435.0]),
    (6000, 3584, 18944, 771.5, [1003.8, 773.8, 917.7, 832.8]),
    (5120, 5120, 17408, 717.9, [960.6, 959.8, 886.6, 791.8]),
    (8192, 5120, 17408, 1121.6, [1566.4, 1467.3, 1274.1, 1598.9]),
]


def test_160_columns_where_they_are_no_slower():
    """A product that comes to this choice (of three weight segments, or without columns that go ahead) takes such a tile only where its time was at
    most 1 % above that of the kernels that it would take otherwise."""
    got = routes([c[:3] for c in MEASURED])
    for (M, N, K, other, wide), r in zip(MEASURED, got):
        assert r["tile"] < 8 or wide[r["tile"] - 8] <= 1.012 * other, (M, N, K, r)
    taken = [r["tile"] for r in got if r["tile"] >= 8]
    assert len(taken) >= 8 and set(taken) == {8, 10, 11}


# rows, weight rows, K, us in one launch and in two (whole rounds of 256x256 tiles, and smaller tiles for the columns left)
MEASURED_AHEAD = [
    (1600, 9728, 896, 48.9, 41.4), (3500, 9728, 896, 95.7, 79.2), (512, 37888, 3584, 151.2, 135.9), (640, 37888, 3584, 183.3, 175.9),
    (640, 28672, 4096, 171.2, 160.4), (640, 34816, 5120, 243.9, 237.6), (6000, 3584, 3584, 170.7, 149.3), (6000, 3584, 18944, 794.7, 677.3),
    (8192, 5120, 17408, 1165.7, 1113.2), (900, 37888, 3584, 266.2, 238.2), (1500, 37888, 3584, 360.2, 344.4), (512, 34816, 5120, 208.8, 164.0),
    (1024, 34816, 5120, 364.7, 305.1), (2048, 34816, 5120, 609.9, 570.7), (6740, 3584, 3584, 180.0, 173.1), (6144, 4096, 14336, 614.9, 617.9),
    (4618, 5120, 5120, 237.8, 230.3), (4880, 5120, 17408, 747.1, 770.0), (5107, 5120, 17408, 749.3, 780.6), (1026, 16384, 2048, 91.2, 82.6),
    (1536, 16384, 2048, 109.7, 102.5), (3328, 16384, 2048, 225.7, 228.5), (6167, 16384, 2048, 402.9, 397.6), (9223, 16384, 2048, 603.1, 606.4),
    (2303, 32000, 3584, 460.3, 452.7), (3820, 32000, 3584, 740.0, 743.0), (5877, 32000, 3584, 1121.4, 1130.5), (8441, 32000, 3584, 1596.5, 1593.3),
]


def test_fp32_results_stay_with_the_tiles():
    """Products that one launch of k_gemm_mid.hip would take, whose sums are of two chains, keep them where the results are fp32."""
    shapes = [c[:3] for c in MEASURED_AHEAD] + [(751, 22016, 2048), (978, 17920, 1536), (1586, 9728, 896)]
    for x, bf, f32 in zip(shapes, routes(shapes), routes(shapes, f32=True)):
        assert f32["ahead"] == (0 if f32["tile"] >= 0 else bf["ahead"]), x
    assert any(bf["ahead"] and not f32["ahead"] for bf, f32 in zip(routes(shapes), routes(shapes, f32=True)))


def test_two_launches_where_they_are_no_slower():
    got = routes([c[:3] for c in MEASURED_AHEAD])
    for (M, N, K, one, two), r in zip(MEASURED_AHEAD, got):
        assert r["ahead"] == 0 or two <= 1.015 * one, (M, N, K, r)
    assert sum(r["ahead"] > 0 for r in got) >= 15


def test_160_columns_have_sound_plans():
    """Their times never fall below the weights' at the rate that they stream, however short K, and few rounds of the chip."""
    r = random.Random(4)
    cases = [(int(2 ** r.uniform(6, 17)), int(2 ** r.uniform(3, 17)), 64 * int(2 ** r.uniform(0, 9))) for _ in range(3000)] + [(50000, 4096, 64), (100000, 4096, 64), (100000, 4096, 128)]
    for (M, N, K), p in zip(cases, routes(cases)):
        if p["wide"] >= 0:
            bm = (128, 192, 256, 320)[p["wide"] - 8]
            rounds = -(-M // bm) * -(-N // 160) / 256
            assert p["wide_us"] >= 2 * N * K / 5.3e6 + 3.99 and rounds <= (2 if bm < 320 else 1 if M < 2048 or 2 * M * K > 8e7 else 4)


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
