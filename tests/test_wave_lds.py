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
