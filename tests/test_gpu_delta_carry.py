"""The delta rule's carry over the pieces of long entries (k_delta.hip delta_carry) through its internal entry: the matrix-core forms (dim 64,
128) and the general one, ragged columns, fresh and kept states, one piece and several."""
import ctypes as C

import pytest
import torch

import gpu_util as G
from qwen_inference_engine_amd import _lib

pytestmark = pytest.mark.gpu
SYMBOL = "_ZN3qie3lay11delta_carryERKNS0_11DeltaCarryPEP12ihipStream_t"


class DeltaCarryP(C.Structure):
    _fields_ = [("spans", C.c_void_p), ("n_spans", C.c_int), ("H", C.c_int), ("dim", C.c_int), ("vdim", C.c_int), ("s_loc", C.c_void_p),
                ("trans", C.c_void_p), ("s_in", C.c_void_p), ("state", C.c_void_p), ("slot_stride", C.c_int64), ("state_off", C.c_int64),
                ("write_state", C.c_int)]


@pytest.mark.parametrize("write", [1, 0])
@pytest.mark.parametrize("dim,vdim", [(64, 32), (64, 7), (128, 128), (128, 33), (96, 40)])
def test_carry(qlib, dim, vdim, write):
    H, off = 3, 5
    spans = [(0, 1, 2, 0), (1, 4, 0, 9), (5, 2, 1, 0), (7, 5, 3, 1)]   # first piece, pieces, slot, first position
    n = 12
    g = torch.Generator("cuda").manual_seed(dim + vdim)

    def t(*shape, scale=1.0):
        return torch.randn(*shape, generator=g, device="cuda") * scale
    loc, trans = t(n, H, dim, vdim), t(n, H, dim, dim, scale=dim ** -0.5)
    stride = H * dim * vdim + 11
    state = t(4, stride)
    sp, s_in, got = torch.tensor(spans, dtype=torch.int32, device="cuda"), torch.full((n, H, dim, vdim), 7.0, device="cuda"), state.clone()
    want_in, want = torch.empty_like(loc, dtype=torch.float64), state.double()
    for first, count, slot, pos in spans:
        s = state[slot, off:off + H * dim * vdim].double().view(H, dim, vdim) * (pos > 0)
        for k in range(first, first + count):
            want_in[k] = s
            s = torch.bmm(trans[k].double(), s) + loc[k].double()
        if write:
            want[slot, off:off + H * dim * vdim] = s.flatten()
    p = DeltaCarryP(sp.data_ptr(), len(spans), H, dim, vdim, loc.data_ptr(), trans.data_ptr(), s_in.data_ptr(), got.data_ptr(), stride, off, write)
    torch.cuda.synchronize()
    G.check(getattr(C.CDLL(_lib.load()._name), SYMBOL)(C.byref(p), None), "delta_carry")
    torch.cuda.synchronize()
    # a step: dim products of size 1 / sqrt(dim) in fp32, one chain: under 1e-5 of values that grow by 1 a piece
    for a, b in ((s_in, want_in), (got, want)):
        assert ((a.double() - b).abs() <= 1e-5 * (1 + b.abs())).all()
    if not write:
        assert torch.equal(got, state)


@pytest.mark.parametrize("share", [1e-6, 1e-3, 1.0])
@pytest.mark.parametrize("dim,vdim", [(64, 40), (128, 128), (96, 40)])
def test_local_states_are_rounded_once(qlib, dim, vdim, share):
    """A piece's products are summed by themselves and added to its local state in one rounding: a state of which little is left after a
    piece (fast decay) costs the local state none of its bits."""
    H, n = 2, 3
    g = torch.Generator("cuda").manual_seed(dim)

    def t(*shape):
        return torch.randn(*shape, generator=g, device="cuda")
    loc, trans, state = t(n, H, dim, vdim), share * dim ** -0.5 * t(n, H, dim, dim), t(1, H, dim, vdim)
    sp, s_in, got = torch.tensor([(0, n, 0, 5)], dtype=torch.int32, device="cuda"), torch.zeros_like(loc), state.clone()
    p = DeltaCarryP(sp.data_ptr(), 1, H, dim, vdim, loc.data_ptr(), trans.data_ptr(), s_in.data_ptr(), got.data_ptr(), H * dim * vdim, 0, 1)
    torch.cuda.synchronize()
    G.check(getattr(C.CDLL(_lib.load()._name), SYMBOL)(C.byref(p), None), "delta_carry")
    torch.cuda.synchronize()
    states = torch.cat([s_in, got])
    assert torch.equal(states[0], state[0])
    for k in range(n):   # each piece from the state that entered it
        m, s = trans[k].double(), states[k].double()
        want, size = torch.bmm(m, s) + loc[k].double(), torch.bmm(m.abs(), s.abs())
        # dim fp32 roundings in the products' chain, each of at most their sum's size; one of the result
        assert ((states[k + 1].double() - want).abs() <= 2.0 ** -24 * (1.001 * want.abs() + dim * size)).all()
