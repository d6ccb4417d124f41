"""CPU: the split-K memory of a stream (csrc/split_pool.hpp), compiled with the host compiler and driven with an allocator that
counts: what a capture was given is never freed before release, what none has seen is, and what is set aside stays below what
is in use."""
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen_inference_engine_amd", "csrc")

DRIVER = r"""
#include "split_pool.hpp"
#include <cstdio>
#include <cstdlib>
#include <map>
// stdin: "t bytes tickets capturing fail" takes memory, "r" releases the pool; stdout: "slab slab_bytes cnt cnt_n" or "none", then live blocks
int main() {
    qie::SplitPool p;
    std::map<size_t, size_t> live;   // fake address -> bytes
    size_t next = 4096;
    int fail = 0;
    auto alloc = [&](size_t n) -> void* {
        if (fail && --fail == 0) return nullptr;
        live[next] = n;
        void* r = (void*)next;
        next += n + 4096;
        return r;
    };
    auto rel = [&](void* q) { if (!live.erase((size_t)q)) { std::printf("freed twice\n"); std::exit(1); } };
    char op;
    while (std::scanf(" %c", &op) == 1) {
        if (op == 'r') {
            p.release(rel);
            std::printf("released %zu\n", live.size());
            continue;
        }
        size_t bytes, tickets;
        int capturing;
        if (std::scanf("%zu %zu %d %d", &bytes, &tickets, &capturing, &fail) != 4) return 2;
        bool ok = p.fits(bytes, tickets);
        if (!ok && !capturing) ok = p.grow(bytes, tickets, alloc, rel);   // as g8_workspace does
        if (ok && capturing) p.held = true;
        if (ok) std::printf("%zu %zu %zu %zu", (size_t)p.slab, p.slab_bytes, (size_t)p.cnt, p.cnt_n);
        else std::printf("none");
        for (auto& b : live) std::printf(" %zu:%zu", b.first, b.second);
        std::printf("\n");
    }
}
"""


@pytest.fixture(scope="module")
def pool(tmp_path_factory):
    d = tmp_path_factory.mktemp("pool")
    (d / "drive.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(d / "drive.cpp"), "-o", str(d / "drive")], check=True)

    def run(ops):
        out = subprocess.run([str(d / "drive")], input="\n".join(ops), text=True, capture_output=True, check=True).stdout
        return [line.split() for line in out.splitlines()]
    return run


def take(bytes_, tickets, capturing=0, fail=0):
    return f"t {bytes_} {tickets} {capturing} {fail}"


def test_captured_memory_stays(pool):
    a, b, c, d, e = pool([take(1000, 10), take(900, 10, 1), take(4000, 8), take(4000, 40), "r"])
    assert a[:4] == b[:4]                                     # the capture got what the eager step had
    live = dict(x.split(":") for x in c[4:])
    assert a[0] in live and a[2] in live and c[0] not in (a[0], a[2])
    live = dict(x.split(":") for x in d[4:])
    assert a[0] in live and a[2] in live and c[0] not in live and c[2] not in live   # the second pair no capture has seen
    assert e == ["released", "0"]


def test_growth_inside_a_capture_is_refused(pool):
    a, b, c = pool([take(1000, 10), take(1001, 10, 1), take(1000, 11, 1)])
    assert a[0] != "none" and b[0] == "none" and c[0] == "none"


@pytest.mark.parametrize("fail", [1, 2])
def test_no_memory(pool, fail):
    a, b, c, d = pool([take(1000, 10), take(5000, 10, 0, fail), take(1000, 10), "r"])
    assert b == ["none"] and c[0] != "none" and d == ["released", "0"]


@pytest.mark.parametrize("seed", range(8))
def test_any_sequence(pool, seed):
    r = random.Random(seed)
    calls = [(int(2 ** r.uniform(4, 20)), int(2 ** r.uniform(0, 10)), int(r.random() < 0.4)) for _ in range(60)]
    out = pool([take(*c) for c in calls] + ["r"])
    held = {}
    for (nb, nt, cap), line in zip(calls, out):
        if line[0] == "none":
            assert cap
            continue
        live = {int(a): int(s) for a, s in (x.split(":") for x in line[4:])}
        slab, sb, cnt, cn = map(int, line[:4])
        assert sb >= nb and cn >= nt and live[slab] == sb and live[cnt] == 4 * cn
        if cap:
            held[slab], held[cnt] = sb, 4 * cn
        assert all(live.get(p) == n for p, n in held.items())          # everything a capture has seen, whole
        aside = {p: n for p, n in live.items() if p not in (slab, cnt)}
        assert set(aside) <= set(held) and sum(aside.values()) < sb + 4 * cn
    assert out[-1] == ["released", "0"]
