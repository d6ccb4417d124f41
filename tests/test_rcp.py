"""CPU: reciprocals refined from an approximation within one ulp (csrc/rcp.hpp) are the IEEE quotients, for every mantissa, from either side."""
import subprocess

from gemm_route import CSRC

DRIVER = r"""
#include "rcp.hpp"
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <initializer_list>
int main() {
    long wrong = 0, ones = 0;
    for (uint32_t e : {127u, 128u, 140u, 252u})   // 1, 2, 2^13, 2^125
        for (uint32_t m = e == 127 ? 0 : 0x7ff000; m < 1u << 23; m++) {
            const uint32_t u = e << 23 | m;
            float d;
            std::memcpy(&d, &u, 4);
            const float want = 1.0f / d;
            for (float r : {want, nextafterf(want, 0.0f), nextafterf(want, 2.0f)}) {
                const bool off = qie::rcp_from(d, r) != want;
                (m == 0x7fffff ? ones : wrong) += off;
            }
        }
    const float inf = INFINITY, nan = NAN;
    std::printf("%ld %ld %d\n", wrong, ones, qie::rcp_from(inf, 0.0f) == 0.0f && qie::rcp_from(nan, nan) != qie::rcp_from(nan, nan));
}
"""


def test_every_mantissa(tmp_path):
    (tmp_path / "drive.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "drive.cpp"), "-o", str(tmp_path / "drive")], check=True)
    wrong, ones, ends = (int(v) for v in subprocess.run([str(tmp_path / "drive")], text=True, capture_output=True, check=True).stdout.split())
    assert wrong == 0 and ones <= 8 and ends == 1
