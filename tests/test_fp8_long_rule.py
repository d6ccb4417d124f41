"""CPU: which kernel takes the long rows of the fp8 decode (csrc/gemm_plan.hpp), compiled with the host compiler."""
import os
import subprocess

from test_gpu_fp8_long_rows import SHAPES

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen_inference_engine_amd", "csrc")

DRIVER = r"""
#include "gemm_plan.hpp"
#include <cstdio>
int main() {
    long M, K, tiles, parts;
    while (std::scanf("%ld %ld %ld %ld", &M, &K, &tiles, &parts) == 4) std::printf("%d\n", (int)qie::d8s::whole_tiles(M, K, tiles, parts, 256));
}
"""
# M, K, N, us of the split-K form, us of whole tiles (Qwen2-7B's and Qwen3-14B's down projections, and sizes on both sides of a round)
MEASURED = [
    (1, 18944, 3584, 18.5, 13.9), (8, 18944, 3584, 19.6, 16.9), (8, 17408, 3072, 16.9, 16.3), (8, 17408, 4096, 19.7, 16.2),
    (1, 17408, 4224, 19.3, 20.0), (8, 17408, 4608, 21.4, 25.0), (1, 17408, 5120, 21.6, 20.8), (8, 17408, 5120, 23.1, 25.6),
    (8, 17408, 6144, 25.9, 27.4), (8, 17408, 8192, 36.1, 28.6), (8, 18944, 6144, 31.3, 29.0), (8, 27648, 4608, 33.7, 37.2),
    (1, 27648, 4608, 33.4, 29.7), (8, 9728, 4608, 14.0, 15.1), (8, 9728, 6144, 16.5, 15.6), (8, 9728, 8704, 20.9, 22.7), (8, 9728, 8192, 20.0, 17.5),
    (8, 5120, 5120, 10.6, 10.3), (1, 5120, 5120, 9.9, 8.7), (8, 5120, 12544, 17.0, 17.8), (8, 2560, 4608, 8.7, 6.7), (8, 2560, 13312, 12.6, 11.8),
]


def test_the_faster_one(tmp_path):
    (tmp_path / "drive.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "drive.cpp"), "-o", str(tmp_path / "drive")], check=True)

    def run(cases):
        text = "\n".join("%d %d %d %d" % (M, K, N // 16, -(-K // 2048)) for M, K, N in cases)
        return [int(v) for v in subprocess.run([str(tmp_path / "drive")], input=text, text=True, capture_output=True, check=True).stdout.split()]
    assert run([c[:3] for c in MEASURED]) == [int(whole < split) for *_, split, whole in MEASURED]
    assert all(run(SHAPES)) and {N // 16 <= 256 for _, _, N in SHAPES} == {False, True}   # those of the GPU test: one tile a workgroup and several
    assert not any(run([(M, 18944, 16 * t) for M in (1, 8) for t in (1, 100, 191)])) and all(run([(M, 18944, 16 * t) for M in (1, 8) for t in (192, 224, 256)]))
