"""Kernels of a few routed rows (k_layered.hip), each through its internal entry: places and gathered rows of up to 256 entries, the grouped
router of up to 64 outputs beside the one of more, products of short rows with and without their gate."""
import ctypes as C

import numpy as np
import pytest
import torch

import gpu_util as G
from qwen_inference_engine_amd import _lib

pytestmark = pytest.mark.gpu
LAY = "_ZN3qie3lay"


class LinearP(C.Structure):
    _fields_ = [("A", C.c_void_p), ("lda", C.c_int64), ("W", C.c_void_p), ("ldw", C.c_int64), ("Y", C.c_void_p), ("ldy", C.c_int64),
                ("M", C.c_int), ("N", C.c_int), ("K", C.c_int), ("batch", C.c_int), ("sA", C.c_int64), ("sW", C.c_int64), ("sY", C.c_int64),
                ("round_a", C.c_int), ("grp_off", C.c_void_p), ("mfma", C.c_int)]


def call(name, *args):
    torch.cuda.synchronize()
    fn = getattr(C.CDLL(_lib.load()._name), LAY + name)
    fn.restype = C.c_int
    G.check(fn(*[C.c_void_p(a.data_ptr()) if isinstance(a, torch.Tensor) else a for a in args]), name)
    torch.cuda.synchronize()


@pytest.mark.parametrize("scored", [False, True])
@pytest.mark.parametrize("T,top,E,W", [(1, 1, 1, 8), (3, 2, 10, 1024), (64, 4, 64, 40), (85, 3, 7, 257), (256, 1, 300, 33)])
def test_places(qlib, T, top, E, W, scored):
    g = torch.Generator("cuda").manual_seed(T)
    sel = torch.randint(0, E, (T * top,), generator=g, device="cuda", dtype=torch.int32)
    y, score = torch.randn(T, W, generator=g, device="cuda"), torch.rand(T * top, generator=g, device="cuda")
    off, slot, xg = sel.new_full((E + 2,), -7), sel.new_full((T * top + 1,), -7), y.new_full((T * top + 1, W), 7.0)
    call("9moe_placeEPKiiiiPiS3_PKfS5_iPfP12ihipStream_t", sel, T, top, E, off, slot, y, score if scored else None, W, xg, None)
    order = torch.argsort(sel, stable=True)
    want = torch.empty_like(sel)
    want[order] = torch.arange(T * top, device="cuda", dtype=torch.int32)
    assert torch.equal(slot[:-1], want) and slot[-1] == -7
    assert off.tolist() == [int((sel < e).sum()) for e in range(E + 1)] + [-7]
    assert torch.equal(xg[:-1], (y.repeat_interleave(top, 0) * (score[:, None] if scored else 1.0))[order]) and (xg[-1] == 7.0).all()


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("E,top,groups,keep", [(1, 1, 1, 1), (10, 2, 1, 1), (24, 5, 6, 2), (64, 64, 1, 1), (64, 8, 8, 3), (72, 8, 8, 3)])
def test_router(qlib, E, top, groups, keep, f32):
    T, W, scale = 5, 136, 1.7
    g = torch.Generator("cuda").manual_seed(E + top)
    y, corr = torch.randn(T, W, generator=g, device="cuda"), 0.1 * torch.randn(E, generator=g, device="cuda")
    w = (torch.randn(E, W, generator=g, device="cuda") * W ** -0.5).to(torch.float32 if f32 else torch.bfloat16)
    sel, score = torch.zeros(T, top, device="cuda", dtype=torch.int32), torch.zeros(T, top, device="cuda")
    call("13route_groupedEPKfPKvS2_biiiiiifPiPfP12ihipStream_t", y, w, corr, C.c_bool(f32), T, W, E, top, groups, keep, C.c_float(scale), sel, score, None)
    s = torch.softmax(y.double() @ w.double().T, 1)
    ch = s + corr.double()
    best = ch.view(T, groups, -1).amax(2)
    drop = best.argsort(1, descending=True)[:, keep:]
    for t in range(T):
        ch[t].view(groups, -1)[drop[t]] = -np.inf
    want = ch.argsort(1, descending=True)[:, :top]
    assert torch.equal(sel.long(), want)   # (the seeds' choices lie further apart than fp32 sums of 136 products)
    chosen = s.gather(1, want)
    assert torch.allclose(score.double(), scale * chosen / chosen.sum(1, keepdim=True), rtol=2e-5)


def test_router_of_many_rows(qlib):
    """Many rows with many choices go to the kernel of one thread a row: the same bits."""
    T, W, E, top = 513, 64, 64, 32
    g = torch.Generator("cuda").manual_seed(2)
    y, corr = torch.randn(T, W, generator=g, device="cuda"), 0.1 * torch.randn(E, generator=g, device="cuda")
    w = torch.randn(E, W, generator=g, device="cuda") * W ** -0.5
    got = []
    for rows in (T, T - 1):
        sel, score = torch.zeros(T, top, device="cuda", dtype=torch.int32), torch.zeros(T, top, device="cuda")
        call("13route_groupedEPKfPKvS2_biiiiiifPiPfP12ihipStream_t", y, w, corr, C.c_bool(True), rows, W, E, top, 4, 3, C.c_float(1.5), sel, score, None)
        got.append((sel[:T - 1], score[:T - 1]))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("K,counts", [(8, [1]), (504, [0, 3, 1]), (512, [2, 0, 0, 5]), (704, [17, 0, 15]), (1024, [1, 1, 0, 2, 2]), (1032, [3, 4])])
def test_short_rows(qlib, K, counts, gated, f32):
    M, E, N = sum(counts), len(counts), 22
    rows = N * (2 if gated else 1)
    g = torch.Generator("cuda").manual_seed(K + M)
    x = torch.randn(M, K, generator=g, device="cuda")
    w = (torch.randn(E, rows, K, generator=g, device="cuda") * K ** -0.5).to(torch.float32 if f32 else torch.bfloat16)
    off = torch.tensor(np.concatenate([[0], np.cumsum(counts)]), dtype=torch.int32, device="cuda")
    y = torch.full((M + 1, N + 3), 7.0, device="cuda")
    p = LinearP(x.data_ptr(), K, w.data_ptr(), K, y.data_ptr(), N + 3, M, N, K, E, 0, rows * K, 0, 0 if f32 else 1, off.data_ptr(), 0)
    done = C.c_bool(True)
    if gated:
        call("12linear_gatedERKNS0_7LinearPEbP12ihipStream_tPb", C.byref(p), C.c_bool(f32), None, C.byref(done))
    else:
        call("6linearERKNS0_7LinearPEbP12ihipStream_t", C.byref(p), C.c_bool(f32), None)
    assert done.value == (K <= 1024 or not gated)
    if not done.value:
        assert (y == 7.0).all()
        return
    xd, e = (x if f32 else x.bfloat16()).double(), torch.repeat_interleave(torch.arange(E, device="cuda"), torch.tensor(counts, device="cuda"))
    z = torch.bmm(w.double()[e].contiguous(), xd[:, :, None]).squeeze(2)
    size = torch.bmm(w.double()[e].abs().contiguous(), xd.abs()[:, :, None]).squeeze(2)
    want, tol = z, 1e-6 * size   # chains of 8 products, 2 and 6 sums: 16 roundings of 6e-8 at most
    if gated:
        a, u = z[:, :N], z[:, N:]
        want = a / (1 + torch.exp(-a)) * u
        # |silu'| <= 1.1, |silu(a)| <= |a|; 4e-7 relative for the gate's own operations
        tol = 1e-6 * (1.1 * size[:, :N] * u.abs() + a.abs() * size[:, N:]) + 1e-12 + 4e-7 * want.abs() * (1 + a.abs())
    assert ((y[:M, :N].double() - want).abs() <= tol).all()
    assert (y[:M, N:] == 7.0).all() and (y[M] == 7.0).all()
