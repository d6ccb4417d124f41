"""Residual add and next norm of the layered models (k_mixers.hip add_norm) through its internal entry: rows on both sides of each register
form's width and past the last, every set of operands, and the routed experts' sum in the branch's place."""
import ctypes as C

import pytest
import torch

import gpu_util as G
from qwen_inference_engine_amd import _lib

pytestmark = pytest.mark.gpu
SYMBOL = "_ZN3qie3lay8add_normEPfPKfS3_S3_S3_S3_S1_PtiifP12ihipStream_tfilRKNS0_9ExpertSumE"


class ExpertSum(C.Structure):
    _fields_ = [("yd", C.c_void_p), ("slot_of", C.c_void_p), ("score", C.c_void_p), ("sel", C.c_void_p), ("y", C.c_void_p),
                ("top", C.c_int), ("n_real", C.c_int)]


def ptr(t):
    return C.c_void_p(t.data_ptr() if t is not None else None)


@pytest.mark.parametrize("W", [5, 256, 1023, 1024, 1025, 2048, 4093, 4096, 4100])
@pytest.mark.parametrize("branch,normed,added,wn", [("", False, True, True), ("v", False, False, True), ("v", True, True, True),
                                                    ("experts", False, False, True), ("identity", True, False, True), ("experts", True, True, False)])
def test_add_norm(qlib, W, branch, normed, added, wn):
    T, top, eps, one = 3, 3, 1e-5, 1.0
    if branch in ("experts", "identity") and W > 4096:
        pytest.skip("longer rows have their sum from a launch of its own")
    g = torch.Generator("cuda").manual_seed(W)

    def t(*shape):
        return torch.randn(*shape, generator=g, device="cuda")
    x, v, add, wb, w, yd, y = t(T, W), t(T, W), t(T, W), 0.1 * t(W), 0.1 * t(W), t(T * top, W), t(T, W)
    score, slot = torch.rand(T * top, generator=g, device="cuda"), torch.randperm(T * top, generator=g, device="cuda").int()
    sel = torch.tensor([0, 4, 1, 5, 2, 3, 1, 0, 2], dtype=torch.int32, device="cuda")
    m, want_v = ExpertSum(), None
    if branch == "v":
        want_v = v.double()
    elif branch:
        rows = yd[slot.long()].double().view(T, top, W)
        if branch == "identity":   # experts 4 and 5 give the row's input
            rows = torch.where((sel >= 4).view(T, top, 1), y.double()[:, None], rows)
        want_v = (score.double().view(T, top, 1) * rows).sum(1)
        m = ExpertSum(yd.data_ptr(), slot.data_ptr(), score.data_ptr(), sel.data_ptr() if branch == "identity" else None, y.data_ptr(), top, 4)
    want = x.double()
    if want_v is not None:
        want = want + (want_v * torch.rsqrt((want_v ** 2).mean(1, keepdim=True) + eps) * (one + wb.double()) if normed else want_v)
    if added:
        want = want + add.double()
    h, h_bf = torch.full((2, T, W), 7.0, device="cuda"), torch.full((T, W), 7.0, device="cuda", dtype=torch.bfloat16)
    xs = x.clone()
    torch.cuda.synchronize()
    fn = getattr(C.CDLL(_lib.load()._name), SYMBOL)
    G.check(fn(ptr(xs), ptr(xs), ptr(v if branch == "v" else None), ptr(wb if normed else None), ptr(add if added else None),
               ptr(w if wn else None), ptr(h), ptr(h_bf), T, W, C.c_float(eps), None, C.c_float(one), 2, C.c_int64(T * W), C.byref(m)), "add_norm")
    torch.cuda.synchronize()
    # a handful of fp32 operations an element, and a mean of W squares (pairs of waves, 16 a lane): under 1e-6 of the operands' size
    assert ((xs.double() - want).abs() <= 2e-6 * (1 + want.abs() + (want_v.abs() if want_v is not None else 0))).all()
    if not wn:
        assert (h == 7.0).all() and (h_bf == 7.0).all()
        return
    out = want * torch.rsqrt((want ** 2).mean(1, keepdim=True) + eps) * (one + w.double())
    assert ((h[0].double() - out).abs() <= 4e-6 * (1 + out.abs())).all() and torch.equal(h[0], h[1])
    assert torch.equal(h_bf, h[0].bfloat16())
