"""The backward kernel's hand-scheduled step loops (head dimensions 128 and 64, both element types, with and
without key intervals per row) where they begin and end: the fewest steps that enter them, row counts around
whole 32-row tiles, several heads per walk, samples and masks whose ends fall inside a token block, and
intervals that cut tiles - against the fp32 oracle."""
import pytest
import torch

from oracle import lvx_oracle as orc
from parity import check_grad

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# (Lq / 32 rounded up) * Hq / Hkv steps a token block; the loops begin at 11 and run 6 steps a trip
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("Hq,Hkv,Lq,Lkv,mask_kind", [
    (4, 1, 65, 128, "none"), (11, 1, 1, 256, "none"), (1, 1, 352, 128, "none"), (4, 2, 257, 200, "none"),
    (4, 1, 95, 130, "kv_len"), (4, 1, 97, 300, "all"), (11, 1, 17, 129, "all"), (8, 1, 300, 500, "images"),
    (4, 1, 600, 700, "images"), (3, 1, 545, 300, "cuts"), (1, 1, 1000, 260, "cuts"), (2, 2, 999, 400, "late")])
def test_backward_loops(D, dtype, Hq, Hkv, Lq, Lkv, mask_kind):
    import lv_xattn
    from lv_xattn import _lib
    _lib.load()
    B, scale = 2, D ** -0.5
    g = torch.Generator().manual_seed(Lq * 1000 + Lkv)
    # memory [B, S, H, D], so that neither rows nor heads lie back to back; what the window's rows are followed
    # by must not be read into a result
    q, do = (torch.randn(B, Lq, Hq, D, generator=g).to(dtype).transpose(1, 2) for _ in range(2))
    k, v = (torch.randn(B, Lkv, Hkv, D, generator=g).to(dtype).transpose(1, 2) for _ in range(2))
    mask, allowed = None, None
    if mask_kind == "kv_len":
        n = torch.tensor([Lkv, Lkv - 70], dtype=torch.int32)
        mask, allowed = lv_xattn.Mask(n), (torch.arange(Lkv) < n[:, None])[:, None].expand(B, Lq, Lkv)
    elif mask_kind != "none":
        row = torch.arange(Lq, dtype=torch.int32).expand(B, Lq)
        if mask_kind == "all":              # every key visible, the ends past the last one
            start, end = torch.zeros_like(row), torch.full_like(row, 2 ** 31 - 1)
        elif mask_kind == "images":         # two images, the second sample has one
            start = torch.where((row >= Lq // 2) & (torch.arange(B)[:, None] == 0), Lkv // 2, 0).int()
            end = start + Lkv // 2
        elif mask_kind == "cuts":           # another interval in every row
            start, end = (row * 7) % (Lkv // 2), Lkv // 2 + (row * 5) % (Lkv // 2)
        else:                               # only rows from the middle on see anything
            start, end = torch.zeros_like(row), torch.where(row >= Lq // 2, Lkv - 3, 0).int()
        start, end = start.contiguous(), end.contiguous()
        n = torch.tensor([Lkv, max(1, Lkv - 70)], dtype=torch.int32)
        mask = lv_xattn.Mask(n, start, end)
        allowed = orc.interval_mask(start.long(), end.long(), Lkv) & (torch.arange(Lkv) < n[:, None])[:, None]
    o, lse = orc.attention_dense(q, k, v, scale, allowed=allowed)
    ref = orc.attention_backward(do, q, k, v, o.to(dtype), lse, scale, allowed=allowed)
    qd, kd, vd, dod = (t.transpose(1, 2).contiguous().to(DEV).transpose(1, 2) for t in (q, k, v, do))
    _, _, _, od, ld = lv_xattn._attn_forward(qd, kd, vd, False, scale, None, rounds=1, mask=mask, batched=True)
    got = lv_xattn._attn_backward(dod, qd, kd, vd, od, ld, False, scale, None, "flash", rounds=1, mask=mask, batched=True)
    torch.cuda.synchronize()
    for name, a, b in zip(("dQ", "dK", "dV"), got, ref):
        check_grad(a, b, name)


# a dense bias joins the loop with intervals per row; the bias of a row is read in chunks of four tokens
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("Hq,Hkv,Lq,Lkv,nb,nh,hidden", [
    (1, 1, 352, 128, 1, 1, "none"), (11, 1, 1, 131, 2, 11, "none"), (4, 2, 257, 202, 1, 4, "none"),
    (4, 1, 97, 300, 2, 1, "none"), (2, 2, 1000, 517, 1, 2, "cuts"), (8, 1, 300, 385, 2, 8, "cuts"),
    (4, 1, 353, 260, 1, 1, "late"), (3, 1, 545, 33, 2, 1, "holes")])
def test_backward_loops_with_a_dense_bias(D, dtype, Hq, Hkv, Lq, Lkv, nb, nh, hidden):
    import lv_xattn
    from lv_xattn import _lib
    _lib.load()
    B, scale = 2, D ** -0.5
    g = torch.Generator().manual_seed(Lq * 1000 + Lkv)
    q, do = (torch.randn(B, Lq, Hq, D, generator=g).to(dtype).transpose(1, 2) for _ in range(2))
    k, v = (torch.randn(B, Lkv, Hkv, D, generator=g).to(dtype).transpose(1, 2) for _ in range(2))
    bias = torch.randn(nb, nh, Lq, Lkv, generator=g)
    row, key = torch.arange(Lq)[:, None], torch.arange(Lkv)
    if hidden == "cuts":                # another interval in every row
        bias.masked_fill_((key < row * 7 % (Lkv // 2)) | (key >= Lkv // 2 + row * 5 % (Lkv // 2)), float("-inf"))
    elif hidden == "late":              # only rows from the middle on see anything
        bias.masked_fill_((row < Lq // 2) | (key >= Lkv - 3), float("-inf"))
    elif hidden == "holes":             # hidden keys between visible ones, which an interval does not tell
        bias.masked_fill_((row + key) % 3 == 1, float("-inf"))
    o, lse = orc.attention_dense(q, k, v, scale, bias=bias)
    ref = orc.attention_backward(do, q, k, v, o.to(dtype), lse, scale, bias=bias)
    qd, kd, vd, dod = (t.transpose(1, 2).contiguous().to(DEV).transpose(1, 2) for t in (q, k, v, do))
    args = (lambda t: t, [bias.to(DEV)], [])
    _, _, _, od, ld = lv_xattn._attn_forward(qd, kd, vd, False, scale, None, *args, rounds=1, batched=True)
    got = lv_xattn._attn_backward(dod, qd, kd, vd, od, ld, False, scale, None, "flash", *args, rounds=1, batched=True)
    torch.cuda.synchronize()
    for name, a, b in zip(("dQ", "dK", "dV"), got, ref):
        check_grad(a, b, name)
