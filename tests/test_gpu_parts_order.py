"""The kernels that sum parts (the fold of key splits, the sum of dQ's fp32 slices) walk (head, sample, row) in shares of
an eighth: several samples, heads that are no multiple of eight, rows and head dimensions at which the last shares are
short or empty.  The reference is the same computation in fp32."""
import pytest
import torch

from parity import check_grad, check_lse, check_o

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Hq,Hkv,D,Lq,Lkv,splits", [
    (1, 1, 1, 16, 1, 700, 3),
    (3, 5, 5, 128, 1, 2000, 40),            # four lanes share the parts of a row
    (3, 6, 2, 64, 33, 1500, 7),             # two
    (2, 9, 3, 32, 300, 900, 2),
    (5, 8, 2, 16, 65, 1100, 4),
    (3, 32, 8, 128, 31, 900, 5),
])
def test_parts_of_several_samples(B, Hq, Hkv, D, Lq, Lkv, splits, dtype):
    import lv_xattn
    g = torch.Generator(device=DEV).manual_seed(Lq * 7 + Lkv)
    q, do = (torch.randn(B, Hq, Lq, D, device=DEV, generator=g).to(dtype) for _ in range(2))
    k, v = (torch.randn(B, Hkv, Lkv, D, device=DEV, generator=g).to(dtype) for _ in range(2))
    qf, kf, vf, dof = (t.float() for t in (q, k, v, do))
    kf, vf = (t.repeat_interleave(Hq // Hkv, 1) for t in (kf, vf))
    s = qf @ kf.transpose(2, 3).contiguous() * D ** -0.5
    lse = torch.logsumexp(s, -1)
    p = torch.exp(s - lse[..., None])
    o = p @ vf
    ds = p * (dof @ vf.transpose(2, 3).contiguous() - (dof * o).sum(-1, keepdim=True))
    dq = ds @ kf * D ** -0.5
    _, _, _, got_o, got_lse = lv_xattn._attn_forward(q, k, v, False, D ** -0.5, "flash", kv_splits=splits)
    got = lv_xattn._attn_backward(do, q, k, v, o.to(dtype), lse.reshape(B * Hq, Lq), False, D ** -0.5, None, "flash")
    torch.cuda.synchronize()
    check_o(got_o.cpu(), o.cpu())
    check_lse(got_lse.cpu().reshape(B, Hq, Lq), lse.cpu())
    check_grad(got[0].cpu(), dq.cpu(), "dQ")
