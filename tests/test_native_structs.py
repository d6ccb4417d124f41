"""CPU: the argument structs that GPU tests hand to internal entry points are csrc/k_layered.hpp's, field by field (the entries' names hold the argument
types, so another signature does not load; another field would be read from the wrong place)."""
import ctypes as C
import os
import re

import pytest

import test_gpu_add_norm
import test_gpu_delta_carry
import test_gpu_delta_walk
import test_gpu_gated_rows
import test_gpu_routed_rows
from gemm_route import CSRC

TYPES = {"int": C.c_int, "int64_t": C.c_int64, "float": C.c_float}


@pytest.mark.parametrize("struct", [test_gpu_add_norm.ExpertSum, test_gpu_delta_carry.DeltaCarryP, test_gpu_delta_walk.DeltaScanP, test_gpu_gated_rows.GatedP,
                                    test_gpu_routed_rows.LinearP], ids=lambda s: s.__name__)
def test_fields(struct):
    text = open(os.path.join(CSRC, "k_layered.hpp")).read()
    (body,) = re.findall(r"^struct %s \{\n(.*?)^\};" % struct.__name__, text, re.S | re.M)
    want = []
    for decl in re.sub(r"//.*", "", body).split(";")[:-1]:
        kind, names = re.fullmatch(r"\s*(?:const )?(\w+(?: ?\*)?) ?(.*?)\s*", decl).groups()
        for name in names.split(","):
            want.append((name.strip(), C.c_void_p if "*" in kind else TYPES[kind]))
    assert [tuple(f) for f in struct._fields_] == want
