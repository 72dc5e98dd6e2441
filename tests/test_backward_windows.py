"""A backward call cuts its rows into windows of unequal length and sizes one workspace for the longest: that
workspace has to serve every other window too, although a window on the other side of a 256-row tile
of the dQ product is cut into another number of partial sums."""
import ctypes as C

import pytest
import torch

from oracle import lvx_oracle as orc
from parity import check_grad

DEV = "cuda:0"


def _bytes(lib, rows, Lq, B, Hq, Hkv, D, Lkv, masked):
    from lv_xattn._lib import AttnShape
    s = AttnShape(B, Hq, Hkv, D, Lq, Lkv, 1, 1.0, None, 0x3000 if masked else None, 0x3100 if masked else None)
    return lib.lvx_bwd_workspace_bytes(C.byref(s), rows)


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,D,Lkv", [(1, 32, 8, 128, 6404), (1, 8, 2, 64, 900), (2, 16, 16, 128, 4096), (1, 1, 1, 16, 129)])
def test_a_longer_window_never_needs_a_smaller_workspace(B, Hq, Hkv, D, Lkv, masked):
    from lv_xattn import _lib
    lib = _lib.load()
    needs = [_bytes(lib, r, 4100, B, Hq, Hkv, D, Lkv, masked) for r in range(1, 2100)]
    assert all(a <= b for a, b in zip(needs, needs[1:]))


@pytest.mark.parametrize("masked", [False, True])
def test_the_longest_window_sizes_the_workspace_of_a_call(masked):
    from lv_xattn import _lib
    from lv_xattn.attn import q_block_bounds
    lib = _lib.load()
    for Lq, rounds in [(513, 2), (4100, 16), (1030, 4), (770, 3), (2049, 8)]:
        rows = [r1 - r0 for r0, r1 in q_block_bounds(Lq, rounds) if r1 > r0]
        needs = [_bytes(lib, r, Lq, 1, 32, 8, 128, 6404, masked) for r in rows]
        assert max(rows) > 256 >= min(rows) and needs[rows.index(max(rows))] == max(needs)


@pytest.mark.gpu
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("Lq,rounds", [(513, 2), (1030, 4), (4100, 16)])
def test_rounds_on_both_sides_of_256_rows(Lq, rounds, masked):
    import lv_xattn
    from lv_xattn.async_communication import reset_global_memory_buffer
    B, Hq, Hkv, D, Lkv = 1, 32, 8, 16, 1024
    g = torch.Generator().manual_seed(Lq)
    q, do = (torch.randn(B, Hq, Lq, D, generator=g).bfloat16() for _ in range(2))
    k, v = (torch.randn(B, Hkv, Lkv, D, generator=g).bfloat16() for _ in range(2))
    mask, allowed = None, None
    if masked:
        row = torch.arange(Lq, dtype=torch.int32).expand(B, Lq)
        start, end = (row * 3 % 500).contiguous(), (500 + row * 5 % 500).contiguous()
        mask, allowed = lv_xattn.Mask(None, start, end), orc.interval_mask(start.long(), end.long(), Lkv)
    o, lse = orc.attention_dense(q, k, v, D ** -0.5, allowed=allowed)
    ref = orc.attention_backward(do, q, k, v, o.bfloat16(), lse, D ** -0.5, allowed=allowed)
    reset_global_memory_buffer()            # no larger workspace of an earlier call in its place
    got = lv_xattn._attn_backward(do.to(DEV), q.to(DEV), k.to(DEV), v.to(DEV), o.bfloat16().to(DEV), lse.to(DEV), False, D ** -0.5,
                                  None, "flash", rounds=rounds, mask=mask)
    torch.cuda.synchronize()
    for name, a, b in zip(("dQ", "dK", "dV"), got, ref):
        check_grad(a, b, name)
