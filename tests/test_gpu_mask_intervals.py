"""lvx_mask_intervals: an additive mask as transformers builds it against the intervals it was made from, at
row lengths and alignments where the 8-byte words of a row begin before it or end behind it, and on
masks that are more than intervals."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,Lq,Lkv,offset", [(1, 1, 1, 0), (2, 3, 7, 0), (3, 4, 1601, 1), (2, 30, 333, 3), (1, 2, 4096, 2)])
def test_mask_intervals(dtype, B, Lq, Lkv, offset):
    from lv_xattn import ops
    g = torch.Generator().manual_seed(Lkv)
    neg = torch.finfo(dtype).min
    start = torch.randint(0, Lkv, (B, Lq), generator=g)
    end = (start + 1 + torch.randint(0, Lkv, (B, Lq), generator=g)).clamp(max=Lkv)
    keys = torch.arange(Lkv)
    visible = (keys >= start[..., None]) & (keys < end[..., None])
    memory = torch.zeros(B * Lq * Lkv + 8, dtype=dtype, device=DEV)
    mask = memory[offset:offset + B * Lq * Lkv].view(B, 1, Lq, Lkv)
    mask.masked_fill_(~visible[:, None].to(DEV), neg)
    got = ops.mask_intervals(mask)
    assert torch.equal(got.kv_start.cpu(), start.int()) and torch.equal(got.kv_end.cpu(), end.int())
    memory[:offset] = 1.0           # what lies before the first row and behind the last is no part of the mask
    memory[offset + B * Lq * Lkv:] = 1.0
    assert ops.mask_intervals(mask) is not None
    finite = mask.clone()
    finite[-1, 0, -1, int(start[-1, -1])] = 0.5
    nothing = mask.clone()
    nothing[0, 0, 0] = neg
    assert ops.mask_intervals(finite) is None and ops.mask_intervals(nothing) is None
    if Lkv > 2:
        gap = torch.zeros_like(mask)
        gap[0, 0, 0, Lkv // 2] = float("-inf")
        assert ops.mask_intervals(gap) is None
