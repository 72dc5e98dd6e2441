"""The product that forms dQ from the dS^T workspace, at the ends of its stages of 32 tokens, tiles of 32 rows and groups
of eight, with one and with several ranges of tokens, against the fp32 oracle: keys and values past a sample's end are NaN,
and so is whatever the backward's kernels do not write of the workspace."""
import pytest
import torch

from oracle import lvx_oracle as orc
from parity import check_grad

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# 40 heads x 2 samples x 2 groups: more work-groups than half the CUs; 10 x 2 x 9: work-groups of 64 rows, one range; the others
# are cut into several
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Hq,Hkv,D,Lq,Lkv,short", [
    (40, 2, 64, 300, 200, 163), (40, 4, 16, 257, 129, 1), (20, 20, 32, 513, 300, 257), (34, 1, 128, 290, 161, 159),
    (10, 2, 128, 513, 300, 257), (8, 8, 64, 1000, 260, 129), (9, 3, 16, 577, 1000, 930),
    (2, 1, 128, 1, 33, 31), (2, 2, 128, 31, 500, 255), (1, 1, 64, 257, 1000, 641), (2, 1, 16, 33, 700, 384), (1, 1, 128, 64, 64, 64)])
def test_dq(Hq, Hkv, D, Lq, Lkv, short, dtype):
    import lv_xattn
    from lv_xattn import async_communication as ac
    B, scale = 2, D ** -0.5
    g = torch.Generator().manual_seed(Lq * 7 + Lkv)
    q, do = (torch.randn(B, Hq, Lq, D, generator=g).to(dtype) for _ in range(2))
    k, v = (torch.randn(B, Hkv, Lkv, D, generator=g).to(dtype) for _ in range(2))
    n = torch.tensor([Lkv, short], dtype=torch.int32)
    allowed = (torch.arange(Lkv) < n[:, None])[:, None].expand(B, Lq, Lkv)
    o, lse = orc.attention_dense(q, k, v, scale, allowed=allowed)
    ref = orc.attention_backward(do, q, k, v, o.to(dtype), lse, scale, allowed=allowed)
    for x in (k, v):
        x[1, :, short:] = float("nan")
    qd, kd, vd, dod, od, ld = (t.to(DEV) for t in (q, k, v, do, o.to(dtype), lse.float()))
    mask = lv_xattn.Mask(n.to(DEV))

    def backward():
        return lv_xattn._attn_backward(dod, qd, kd, vd, od, ld, False, scale, None, "flash", rounds=1, mask=mask, batched=True)

    backward()
    for key, buf in ac._WORKSPACES.items():
        if key[0] == "bwd_ds":
            buf.fill_(0xff)
    got = backward()
    torch.cuda.synchronize()
    for name, a, b in zip(("dQ", "dK", "dV"), got, ref):
        check_grad(a, b, name)
