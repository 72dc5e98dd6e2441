"""The native operators let other Python threads run while they launch."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def test_launches_do_not_hold_the_interpreter_lock():
    """In the place of the library's functions: the interpreter's own PyGILState_Check, which answers 1 - an error
    code - to a thread that holds the lock, and launches nothing."""
    from lv_xattn import _lib, ops
    host = _lib.host()
    q, o, do, dq = (torch.zeros(1, 4, 8, 128, device=DEV, dtype=torch.bfloat16) for _ in range(4))
    k, v, dk, dv = (torch.zeros(1, 1, 16, 128, device=DEV, dtype=torch.bfloat16) for _ in range(4))
    lse, delta = (torch.zeros(4, 8, device=DEV) for _ in range(2))
    ws = torch.zeros(1 << 20, device=DEV, dtype=torch.uint8)
    held = ctypes.cast(ctypes.pythonapi.PyGILState_Check, ctypes.c_void_p).value
    assert ctypes.pythonapi.PyGILState_Check() == 1
    host.bind({name: held for name in _lib.SYMBOLS})
    try:
        ops.fwd(q, k, v, o, lse, 0.1)
        ops.fwd(q, k, v, o, lse, 0.1, acc=(do, delta))
        ops.bwd_preprocess(o, do, delta)
        ops.bwd(q, k, v, do, lse, delta, dq, dk, dv, 0.1, workspace=ws)
    finally:
        _lib._host_lib = None
        _lib.host()


class _Declines:
    """A native side that passes no call on: the operators go through their own checks and ctypes."""
    def __getattr__(self, name):
        return lambda *a: None if name == "bias_hull" else -1 if name == "bwd_workspace_bytes" else False


def _bias(nb, nh, Lq, Lkv, seed):
    pad = -Lkv % 4
    b = torch.randn(nb, nh, Lq, Lkv + pad, generator=torch.Generator().manual_seed(seed))
    b[..., ::3] = -torch.inf
    b[..., Lkv // 2:] = -torch.inf
    return b.to(DEV)[..., :Lkv]


@pytest.mark.parametrize("B,H,nb,nh,Lq,Lkv", [(1, 4, 1, 1, 1, 130), (2, 4, 1, 4, 33, 257), (2, 4, 2, 1, 64, 1024), (3, 8, 3, 8, 5, 63)])
def test_a_dense_bias_goes_the_same_way_natively(monkeypatch, B, H, nb, nh, Lq, Lkv):
    from lv_xattn import ops
    g = torch.Generator().manual_seed(Lkv)
    q, do, o = (torch.randn(B, H, Lq, 64, generator=g).to(DEV, torch.float16) for _ in range(3))
    k, v = (torch.randn(B, 2, Lkv, 64, generator=g).to(DEV, torch.float16) for _ in range(2))
    bias = _bias(nb, nh, Lq, Lkv, Lq)
    ws = torch.empty(ops.bwd_workspace_bytes(q, k, Lq, ops.bias_hull(q, k, bias)), dtype=torch.uint8, device=DEV)

    def results():
        hull = ops.bias_hull(q, k, bias)
        out, lse, delta = torch.empty_like(q), torch.empty(B * H, Lq, device=DEV), torch.empty(B * H, Lq, device=DEV)
        ops.fwd(q, k, v, out, lse, 0.125, mask=hull, bias=bias)
        ops.bwd_preprocess(out, do, delta)
        dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
        ops.bwd(q, k, v, do, lse, delta, dq, dk, dv, 0.125, mask=hull, workspace=ws, bias=bias)
        return hull.kv_start, hull.kv_end, out, lse, dq, dk, dv, torch.tensor(ops.bwd_workspace_bytes(q, k, Lq, hull))

    native = results()
    monkeypatch.setattr(ops, "host", _Declines)
    for a, b in zip(native, results()):
        assert torch.equal(a, b)


def test_a_bias_the_library_cannot_read_is_refused():
    from lv_xattn import ops
    from lv_xattn._lib import LvxError
    q, o = (torch.zeros(1, 4, 8, 64, device=DEV, dtype=torch.float16) for _ in range(2))
    k = torch.zeros(1, 2, 30, 64, device=DEV, dtype=torch.float16)
    lse = torch.zeros(4, 8, device=DEV)
    good = _bias(1, 1, 8, 30, 0)
    for bad in (good.contiguous(), good.double(), good.cpu(), good[:, :, :7], good.expand(3, 1, 8, 30), good[0]):
        with pytest.raises(LvxError):
            ops.fwd(q, k, k, o, lse, 0.1, bias=bad)
        with pytest.raises(LvxError):
            ops.bias_hull(q, k, bad)
