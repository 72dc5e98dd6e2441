"""Which dS^T tiles an interval mask leaves alive: masks whose intervals change at, beside and far inside the 256-row
groups of the dQ contraction and in more runs than a token block keeps, against the fp32 oracle, with a workspace of NaN
(a tile that nobody wrote must not be read)."""
import pytest
import torch

from oracle import lvx_oracle as orc
from parity import check_grad

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _intervals(kind, B, Lq, Lkv):
    row = torch.arange(Lq).expand(B, Lq)
    if kind == "every_32":              # another quarter of the keys in every row tile: a run per fourth tile
        lo = (row // 32 % 4) * (Lkv // 4)
        return lo, lo + Lkv // 4
    if kind == "inside":                # two images, the second from a row inside a group, another in each sample
        second = row >= 97 + 140 * torch.arange(B)[:, None]
        lo = torch.where(second, Lkv // 2, 0)
        return lo, lo + Lkv // 2
    if kind == "holes":                 # whole tiles of rows that see nothing, and single rows that see all
        sees = (row // 32 % 3 == 1) | (row % 61 == 60)
        return torch.zeros_like(row), torch.where(sees, torch.where(row % 61 == 60, Lkv, 200), 0)
    hi = 1 + (row * 131 + 17) % Lkv     # "random": ends of every length
    return (hi * 3) // 5, hi


@pytest.mark.parametrize("rounds,batched", [(1, True), (3, False)])
@pytest.mark.parametrize("Hq,Hkv,D,Lq,Lkv", [(2, 1, 128, 600, 1100), (2, 2, 64, 511, 700), (1, 1, 128, 2700, 520), (3, 1, 32, 290, 390)])
@pytest.mark.parametrize("kind", ["every_32", "inside", "holes", "random"])
def test_live_tiles(kind, Hq, Hkv, D, Lq, Lkv, rounds, batched):
    import lv_xattn
    from lv_xattn import async_communication as ac
    B, scale = 2, D ** -0.5
    g = torch.Generator().manual_seed(Lq + Lkv)
    q, do = (torch.randn(B, Hq, Lq, D, generator=g).bfloat16() for _ in range(2))
    k, v = (torch.randn(B, Hkv, Lkv, D, generator=g).bfloat16() for _ in range(2))
    start, end = (t.int().contiguous() for t in _intervals(kind, B, Lq, Lkv))
    n = torch.tensor([Lkv, Lkv - 150], dtype=torch.int32)
    allowed = orc.interval_mask(start.long(), end.long(), Lkv) & (torch.arange(Lkv) < n[:, None])[:, None]
    o, lse = orc.attention_dense(q, k, v, scale, allowed=allowed)
    ref = orc.attention_backward(do, q, k, v, o.bfloat16(), lse, scale, allowed=allowed)
    qd, kd, vd, dod = (t.to(DEV) for t in (q, k, v, do))
    mask = lv_xattn.Mask(n.to(DEV), start.to(DEV), end.to(DEV))

    def both():
        _, _, _, od, ld = lv_xattn._attn_forward(qd, kd, vd, False, scale, None, rounds=rounds, mask=mask, batched=batched)
        return lv_xattn._attn_backward(dod, qd, kd, vd, od, ld, False, scale, None, "flash", rounds=rounds, mask=mask, batched=batched)

    both()
    for key, buf in ac._WORKSPACES.items():
        if key[0] == "bwd_ds":
            buf.fill_(0xff)
    got = both()
    torch.cuda.synchronize()
    for name, a, b in zip(("dQ", "dK", "dV"), got, ref):
        check_grad(a, b, f"{name} ({kind})")
