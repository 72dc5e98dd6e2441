"""The hull of a dense bias at the sizes where a row is read from both ends inwards: what the ends hide, in one head or another."""
import pytest
import torch

DEV = "cuda:0"


@pytest.mark.gpu
@pytest.mark.parametrize("Lq,Lkv", [(600, 1025), (520, 1500), (513, 2052), (700, 4099), (600, 6404), (513, 1024)])
@pytest.mark.parametrize("B,H", [(1, 1), (2, 3)])
def test_every_row_has_the_span_of_what_it_sees(B, H, Lq, Lkv):
    from lv_xattn import ops
    g = torch.Generator(device=DEV).manual_seed(Lkv + H)
    bias = torch.zeros(B, H, Lq, (Lkv + 3) // 4 * 4, device=DEV)[..., :Lkv]
    at = torch.arange(Lkv, device=DEV)
    lo = torch.randint(0, Lkv, (B, H, Lq, 1), generator=g, device=DEV)
    n = torch.randint(0, Lkv, (B, H, Lq, 1), generator=g, device=DEV)
    lo[..., ::3, :], n[..., ::5, :] = lo[..., ::3, :] % 300, Lkv
    n[..., 7, :] = 0                                # nothing
    n[..., 8, :], lo[..., 8, :] = 1, Lkv - 1        # the last key
    n[..., 9, :], lo[..., 9, :] = 1, 0
    bias.masked_fill_((at < lo) | (at >= lo + n), -float("inf"))
    bias.masked_fill_((torch.rand(bias.shape, generator=g, device=DEV) < 0.3) & (n < Lkv), -float("inf"))
    seen = (bias != -float("inf")).any(1)
    some = seen.any(-1)
    start = torch.where(some, seen.int().argmax(-1), 0)
    end = torch.where(some, Lkv - seen.flip(-1).int().argmax(-1), 0)
    q, k = (torch.zeros(B, 3 if H == 3 else 2, L, 16, dtype=torch.float16, device=DEV) for L in (Lq, Lkv))
    hull = ops.bias_hull(q, k, bias)
    assert torch.equal(hull.kv_start.long(), start) and torch.equal(hull.kv_end.long(), end)
