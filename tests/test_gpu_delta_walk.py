"""The gated delta rule in order over entries of many rows (k_delta.hip delta_walk) through its internal entry, against the rule in 64 bits: heads that fill
their lanes and not, ragged columns, decay by head and by channel, lengths about the 16 rows that are staged at a time, fresh and kept states."""
import ctypes as C

import pytest
import torch

import gpu_util as G
from qwen_inference_engine_amd import _lib

pytestmark = pytest.mark.gpu


class DeltaScanP(C.Structure):
    _fields_ = [("qkv", C.c_void_p), ("ld_qkv", C.c_int64), ("beta", C.c_void_p), ("ld_beta", C.c_int64), ("g", C.c_void_p), ("ld_g", C.c_int64),
                ("entries", C.c_void_p), ("n_entries", C.c_int), ("H", C.c_int), ("G", C.c_int), ("dim", C.c_int), ("vdim", C.c_int), ("state", C.c_void_p),
                ("slot_stride", C.c_int64), ("state_off", C.c_int64), ("read_state", C.c_int), ("write_state", C.c_int), ("out", C.c_void_p),
                ("trans", C.c_void_p), ("w_out", C.c_void_p)]


def run(name, p):
    torch.cuda.synchronize()
    G.check(getattr(C.CDLL(_lib.load()._name), "_ZN3qie3lay10%sERKNS0_10DeltaScanPEP12ihipStream_t" % name)(C.byref(p), None), name)
    torch.cuda.synchronize()


@pytest.mark.parametrize("read,write", [(1, 1), (0, 0), (2, 1)])
@pytest.mark.parametrize("head", [True, False])
@pytest.mark.parametrize("dim,vdim", [(8, 1), (24, 40), (64, 64), (72, 15), (96, 17), (128, 128)])
def test_walk(qlib, dim, vdim, head, read, write):
    H, K, off, lens = 4, 2, 5, [1, 15, 16, 17, 33, 200]
    entries, T = [], 3   # (rows of no entry before the first)
    for i, n in enumerate(lens):
        entries.append((T, n, len(lens) - 1 - i, 7 * (i % 2)))
        T += n
    gen = torch.Generator("cuda").manual_seed(dim + vdim)

    def t(*shape):
        return torch.randn(*shape, generator=gen, device="cuda")
    ld = (2 * K * dim + H * vdim + 3) // 4 * 4
    qkv = t(T, ld)
    q, k = qkv[:, :K * dim].view(T, K, dim), qkv[:, K * dim:2 * K * dim].view(T, K, dim)
    q.div_(q.norm(dim=-1, keepdim=True) * dim ** 0.5)
    k.div_(k.norm(dim=-1, keepdim=True))
    v = qkv[:, 2 * K * dim:2 * K * dim + H * vdim].view(T, H, vdim)
    beta, g = torch.rand(T, H + 1, generator=gen, device="cuda"), torch.rand(T, H * (1 if head else dim), generator=gen, device="cuda") ** 0.1
    stride = H * dim * vdim + 11
    start = t(len(lens), stride)
    ent = torch.tensor(entries, dtype=torch.int32, device="cuda")
    err = {}
    for name in ("delta_walk", "delta_scan"):
        state, out = start.clone(), torch.full((T, H, vdim), 7.0, device="cuda")
        run(name, DeltaScanP(qkv.data_ptr(), ld, beta.data_ptr(), H + 1, g.data_ptr(), H if head else 0, ent.data_ptr(), len(lens), H, K, dim, vdim,
                             state.data_ptr(), stride, off, read, write, out.data_ptr(), None, None))
        want_state, worst, sums = start.double(), 0.0, [0.0, 0.0]
        assert (out[:3] == 7.0).all()
        for first, n, slot, pos in entries:
            s = start[slot, off:off + H * dim * vdim].double().view(H, dim, vdim) * (1.0 if read == 2 or (read == 1 and pos > 0) else 0.0)
            want = torch.empty(n, H, vdim, dtype=torch.float64, device="cuda")
            for i in range(n):
                r = first + i
                kk, qq = (x[r].double().repeat_interleave(H // K, 0).unsqueeze(-1) for x in (k, q))
                s = s * g[r].double().view(H, -1, 1)
                u = beta[r, :H].double().view(H, 1) * (v[r].double() - (s * kk).sum(1))
                s = s + kk * u.unsqueeze(1)
                want[i] = (s * qq).sum(1)
            d = out[first:first + n].double() - want
            sums[0] += float((d ** 2).sum())
            sums[1] += float((want ** 2).sum())
            # a row adds some dim roundings of 6e-8 of values of order 1, which the decays and the rule itself forget: under 1e-5
            assert (d.abs() <= 1e-5 * (1 + want.abs())).all()
            if write:
                want_state[slot, off:off + H * dim * vdim] = s.flatten()
        assert ((state.double() - want_state).abs() <= 1e-5 * (1 + want_state.abs())).all()
        err[name] = (sums[0] / sums[1]) ** 0.5
    print("error against 64 bits: %.3g, of the scan %.3g" % (err["delta_walk"], err["delta_scan"]))
    assert err["delta_walk"] <= 1.1 * err["delta_scan"] + 1e-9
