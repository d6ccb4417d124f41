"""The GEMM dispatch's host rules (csrc/gemm_plan.hpp), compiled with the host compiler: which kernel and tile a product takes."""
import os
import subprocess
import tempfile

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen_inference_engine_amd", "csrc")

DRIVER = r"""
#include "gemm_plan.hpp"
#include <cstdio>
int main() {
    long M, cols, K, gated, ragged, cus, f32;
    while (std::scanf("%ld %ld %ld %ld %ld %ld %ld", &M, &cols, &K, &gated, &ragged, &cus, &f32) == 7) {
        const qie::mid::Plan p = qie::mid::choose(M, cols, K, cus), w = qie::mid::plan_wide(M, cols, K, cus);
        const long ahead = (long)qie::mid::columns_ahead(M, cols, K, cus, f32 != 0);
        const qie::mid::Plan r = qie::mid::best(M, ahead > 0 ? cols - ahead : cols, K, cus);
        const int few = qie::few::choose(M, cols, K, cus, gated != 0, ragged != 0).form;
        std::printf("%d %d %d %d %d %d %d %d %ld %d %d %.9g\n", p.tile, few, few >= 0 ? -2 : p.tile, p.n_mt * p.n_nt, p.splitk, p.whole, qie::g8p::parts(M, cols, K, cus), w.tile, ahead,
                    ahead > 0 ? r.tile : -1, ahead > 0 ? r.splitk : 0, w.us);
    }
}
"""


def routes(cases, cus=256, f32=False):
    """For every (rows, weight rows, K), or (.., gate and up, weight segments that are no multiples of 64 rows): {mid (k_gemm_mid.hip's tile where it is
    asked: numbers of mid::TILES and mid::WIDE, -1: none), few (k_gemm_few.hip's form, asked before that, -1: none), tile (mid, or -2: few has it),
    tiles, splitk, whole (tiles that are not split), parts (of the 256x256 kernel, 0: not its launch; taken where tile is -1), wide (the best 160-column
    tile), ahead (columns that the 256x256 kernel takes of a product of one weight segment, with f32 of one with fp32 results, or gate and up, with the
    other columns in a launch behind it; 0: the one launch above), rest, rest_splitk (that launch's tile and parts), wide_us}."""
    with tempfile.TemporaryDirectory() as d:
        src, exe = os.path.join(d, "drive.cpp"), os.path.join(d, "drive")
        with open(src, "w") as f:
            f.write(DRIVER)
        subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, src, "-o", exe], check=True)
        text = "\n".join("%d %d %d %d %d %d %d" % (*c, *(0, 0)[len(c) - 3:], cus, f32) for c in cases)
        out = subprocess.run([exe], input=text, text=True, capture_output=True, check=True).stdout
    names = ("mid", "few", "tile", "tiles", "splitk", "whole", "parts", "wide", "ahead", "rest", "rest_splitk", "wide_us")
    return [dict(zip(names, [int(v) for v in line.split()[:-1]] + [float(line.split()[-1])])) for line in out.splitlines()]
