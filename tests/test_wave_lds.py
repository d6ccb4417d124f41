"""CPU: exchanges through LDS between the lanes of a wave.  __builtin_amdgcn_wave_barrier() holds the wave's order but is no memory fence to
the compiler, which may move a lane's read of another's value ahead of the write; every use stands between a release and an acquire."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen_inference_engine_amd", "csrc")


def test_wave_barriers_stand_between_fences():
    found = 0
    for path in glob.glob(os.path.join(CSRC, "*.h*")):
        lines = open(path).read().splitlines()
        for i, line in enumerate(lines):
            if re.match(r"\s*__builtin_amdgcn_wave_barrier\(\);", line):
                found += 1
                assert "__builtin_amdgcn_fence(__ATOMIC_RELEASE" in lines[i - 1], f"{path}:{i + 1}"
                assert "__builtin_amdgcn_fence(__ATOMIC_ACQUIRE" in lines[i + 1], f"{path}:{i + 1}"
    assert found


FENCE = re.compile(r"__syncthreads\(\)|wave_lds_fence\(\)|__builtin_amdgcn_s_barrier\(\)")


def test_transposing_reads_stand_between_fences():
    """Every ds_read_b64_tr_b16 reads what other lanes wrote: a fence or barrier stands between the last write to that array before it and the
    read, and between the read and the next write to the array, under its own name or another pointer's."""
    found = 0
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h*"))):
        text = open(path).read()
        for at in re.finditer(r"__builtin_amdgcn_ds_read_tr16_b64_v4i16\(\s*\(__attribute__\(\(address_space\(3\)\)\) i16x4_t\*\)\s*\(+(\w+)", text):
            found += 1
            array = at.group(1)
            alias = re.findall(rf"uint16_t\* {array} = (\w+) \+", text[:at.start()])
            array = alias[-1] if alias else array
            names = {array} | set(re.findall(rf"\* (\w+) = reinterpret_cast<\w+\*>\({array}\)", text))
            writes = [m.start() for m in re.finditer(r"(?:reinterpret_cast<[\w ]+\*>\(|\b)(?:%s)(?: \+ [^;=]*\)|\[[^;=]*\]) = " % "|".join(names), text)]
            for w in [w for w in writes if w < at.start()][-1:]:
                assert FENCE.search(text, w, at.start()), f"{path}: write of {array} before {text.count(chr(10), 0, at.start()) + 1}"
            for w in [w for w in writes if w > at.start()][:1]:
                assert FENCE.search(text, at.start(), w), f"{path}: write of {array} behind {text.count(chr(10), 0, at.start()) + 1}"
            print(os.path.basename(path), array, sorted(names), [text.count("\n", 0, w) + 1 for w in writes])
    assert found >= 4
