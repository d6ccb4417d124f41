"""The prompts' attention dispatch (csrc/attn_plan.hpp), compiled with the host compiler: which form of the kernel a call takes."""
import os
import subprocess
import tempfile

from gemm_route import CSRC

DRIVER = r"""
#include "attn_plan.hpp"
#include <cstdio>
int main() {
    long rows, heads, hd;
    while (std::scanf("%ld %ld %ld", &rows, &heads, &hd) == 3) {
        const qie::PrefillAttnPlan p = qie::prefill_attn_plan_of(rows, heads, (int)hd, 256);
        std::printf("%d %d\n", p.waves, p.groups);
    }
}
"""


def forms(cases):
    """For every (rows of a sequence, sequences, heads, head size): (waves of a workgroup, 16-row groups of a wave)."""
    with tempfile.TemporaryDirectory() as d:
        src, exe = os.path.join(d, "drive.cpp"), os.path.join(d, "drive")
        with open(src, "w") as f:
            f.write(DRIVER)
        subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, src, "-o", exe], check=True)
        text = "\n".join("%d %d %d" % (rows, seqs * heads, hd) for rows, seqs, heads, hd in cases)
        out = subprocess.run([exe], input=text, text=True, capture_output=True, check=True).stdout
    return [tuple(int(v) for v in line.split()) for line in out.splitlines()]
