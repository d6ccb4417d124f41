"""CPU: which bytes of x and of the weights k_gemm_few.hip's loads may touch.  The hardware's range check is documented for a lane's offset alone, so by
few::bytes_of and few::row_at (csrc/gemm_plan.hpp) that offset lies in the rows that exist or behind the buffer's end; the scalar offset is a chunk's k."""
import os
import re
import subprocess

from gemm_route import CSRC

DRIVER = r"""
#include "gemm_plan.hpp"
#include <cstdio>
// rows that exist, rows of the tile, row stride, K, first k of the chunk: every 16 bytes that a tile's loads ask for
int main() {
    long rows, tile, ld, K, k;
    while (std::scanf("%ld %ld %ld %ld %ld", &rows, &tile, &ld, &K, &k) == 5) {
        const long bytes = qie::few::bytes_of((int)rows, ld, K), tensor = ((rows - 1) * ld + K) * 2;
        long wrong = 0, read = 0;
        for (int r = 0; r < tile; r++)
            for (int piece = 0; piece < 8; piece++) {
                const long at = (long)qie::few::row_at(r, ld) + 16 * piece, from = 2 * k + at;
                const bool in = at + 16 <= bytes;   // without k: what the check is documented to see
                read += in;
                wrong += in != (r < rows) || (in && (from != 2 * (r * ld + k) + 16 * piece || from + 16 > tensor)) || (!in && at < bytes);
            }
        std::printf("%ld %ld\n", wrong, read);
    }
}
"""


def test_rows_that_do_not_exist_are_not_read(tmp_path):
    (tmp_path / "drive.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "drive.cpp"), "-o", str(tmp_path / "drive")], check=True)
    # (the largest stride that the kernel takes: mid::strides_fit)
    cases = [(rows, tile, ld, K, k) for tile in (16, 32, 64) for rows in {1, 8, 9, tile - 1, tile} for ld, K in ((64, 64), (896, 896), (1000, 896), (1 << 22, 3584))
             for k in {0, K // 128 * 64, K - 64}]
    out = subprocess.run([str(tmp_path / "drive")], input="\n".join("%d %d %d %d %d" % c for c in cases), text=True, capture_output=True, check=True).stdout
    for c, line in zip(cases, out.splitlines(), strict=True):
        assert [int(v) for v in line.split()] == [0, 8 * c[0]], c


def test_scalar_offsets_are_chunks():
    text = open(os.path.join(CSRC, "k_gemm_few.hip")).read()
    calls = re.findall(r"buffer_lds16<.*;", text)
    assert len(calls) == 2 and all(re.search(r", [aw]_at\[b\], k\);$", c) for c in calls) and "raw_ptr_buffer_load_lds" not in text, calls
