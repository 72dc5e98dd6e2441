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
