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


def _shape_of(B, Hq, Hkv, D, rows, Lkv):
    from lv_xattn._lib import AttnShape
    return AttnShape(B, Hq, Hkv, D, rows, Lkv, 1, 1.0, None, None, None)


@pytest.mark.parametrize("B,Hq,Hkv,rows,Lkv,D,mb", [
    (1, 32, 8, 256, 700, 128, 44), (4, 32, 8, 64, 700, 128, 45), (1, 8, 8, 1, 128, 128, 2), (1, 32, 8, 256, 6404, 128, 194)])
def test_windows_too_short_to_be_cut_have_no_room_for_sums_of_ranges(B, Hq, Hkv, rows, Lkv, D, mb):
    from lv_xattn import _lib
    lib, s = _lib.load(), _shape_of(B, Hq, Hkv, D, rows, Lkv)
    need = lib.lvx_bwd_workspace_bytes(C.byref(s), rows)
    assert need == lib.lvx_bwd_acc_workspace_bytes(C.byref(s), rows) <= mb * 10 ** 6


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,D,Lkv", [(1, 32, 8, 128, 1601), (1, 32, 8, 128, 6404), (2, 16, 4, 64, 900), (3, 8, 8, 32, 4000), (1, 2, 1, 16, 129)])
def test_the_room_for_sums_of_ranges(B, Hq, Hkv, D, Lkv, masked):
    """At most 96 ranges an XCD, none in a call that accumulates; that room is the least that any call takes."""
    from lv_xattn import _lib
    lib = _lib.load()
    s = _shape_of(B, Hq, Hkv, D, 4100, Lkv)
    if masked:
        s.kv_start, s.kv_end = 0x3000, 0x3100
    both = [(lib.lvx_bwd_workspace_bytes(C.byref(s), r), lib.lvx_bwd_acc_workspace_bytes(C.byref(s), r)) for r in range(1, 4100, 17)]
    assert all(0 <= full - acc <= 8 * 96 * 2 * 128 * D * 4 for full, acc in both)
    assert all(x[1] <= y[1] for x, y in zip(both, both[1:]))
    t = _lib.Tensor4(0x1000, 4100 * Hq * D, 4100 * D, D)

    def call(ws, room):         # refused for its size, or only then for its address
        return lib.lvx_bwd(C.byref(s), *[C.byref(t)] * 4, 0x2000, 0x2000, *[C.byref(t)] * 3, 0, 0, 4100, ws, room, None)
    least = lib.lvx_bwd_acc_workspace_bytes(C.byref(s), 4100)
    assert (call(0x4000, least - 1), call(0x4001, least)) == (-7, -2)


@pytest.mark.gpu
def test_a_cap_that_holds_all_but_the_sums_of_ranges_leaves_one_window():
    import lv_xattn
    from lv_xattn import async_communication as ac
    from lv_xattn import ops
    B, Hq, Hkv, Lq, Lkv, D = 1, 16, 8, 1024, 1346, 128
    g = torch.Generator(device=DEV).manual_seed(3)
    q, do = (torch.empty(B, Hq, Lq, D, dtype=torch.bfloat16, device=DEV).normal_(generator=g) for _ in range(2))
    k, v = (torch.empty(B, Hkv, Lkv, D, dtype=torch.bfloat16, device=DEV).normal_(generator=g) for _ in range(2))
    o, lse = lv_xattn._attn_forward(q, k, v, False, D ** -0.5, None, rounds=1, batched=True)[3:]
    want = lv_xattn._attn_backward(do, q, k, v, o, lse, False, D ** -0.5, None, "flash", rounds=1, batched=True)
    least, full = (ops.bwd_workspace_bytes(q, k, Lq, accumulate_dkv=a) for a in (True, False))
    assert least < full
    calls, bwd, cap = [], ops.bwd, ac.backward_workspace_cap()
    try:
        ac._BWD_WS_CAP = least
        ops.bwd = lambda *a, **kw: (calls.append((a[10], a[11], kw["accumulate_dkv"], kw["workspace"].numel())), bwd(*a, **kw))[1]
        got = lv_xattn._attn_backward(do, q, k, v, o, lse, False, D ** -0.5, None, "flash", rounds=1, batched=True)
    finally:
        ops.bwd, ac._BWD_WS_CAP = bwd, cap
    assert calls == [(0, Lq, False, least)]
    assert torch.equal(got[0], want[0])
    for a, b in zip(got[1:], want[1:]):         # the same sums, in another order, rounded once
        assert (a.float() - b.float()).norm() <= 4e-3 * b.float().norm()
