"""The backward's first launch: delta formed from O, the zeroed scratch and the tables of an interval mask in one, against the launches
of their own that it stands for."""
import pytest
import torch

DEV = "cuda:0"


def _data(B, Hq, Hkv, Lq, Lkv, D, dtype, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    q, do = (torch.empty(B, Lq, Hq, D, dtype=dtype, device=DEV).normal_(generator=g).transpose(1, 2) for _ in range(2))
    k, v = (torch.empty(B, Hkv, Lkv, D, dtype=dtype, device=DEV).normal_(generator=g) for _ in range(2))
    return q, k, v, do, g


def _intervals(B, Lq, Lkv, g):
    from lv_xattn import Mask
    start = torch.randint(0, Lkv, (B, Lq), generator=g, device=DEV, dtype=torch.int32)
    end = start + torch.randint(0, Lkv // 2, (B, Lq), generator=g, device=DEV, dtype=torch.int32)
    return Mask(None, start, end.clamp(max=Lkv))


def _backward(q, k, v, o, do, lse, mask=None, from_o=True, rounds=1, rows=None):
    from lv_xattn import ops
    B, Hq, Lq, D = q.shape
    r0, n = rows or (0, Lq)
    dq = torch.zeros_like(q)
    kv = dict(dtype=torch.float32 if rounds > 1 else q.dtype, device=DEV)
    dk, dv = (torch.zeros(B, k.shape[2], k.shape[1], D, **kv).transpose(1, 2) for _ in range(2))
    ws = torch.full((ops.bwd_workspace_bytes(q, k, -(-n // rounds), mask),), 0xff, dtype=torch.uint8, device=DEV)
    delta = None
    if not from_o:
        delta = torch.empty(B * Hq, Lq, device=DEV)
        ops.bwd_preprocess(o, do, delta)
    ops.bwd(q, k, v, do, lse, delta, dq, dk, dv, D ** -0.5, r0, n, mask, accumulate_dkv=rounds > 1, workspace=ws, rounds=rounds,
            o=o if from_o else None)
    return dq, dk, dv


def _forward(q, k, v, mask):
    import lv_xattn
    return lv_xattn._attn_forward(q, k, v, False, q.shape[-1] ** -0.5, None, rounds=1, batched=True, mask=mask)[3:]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [128, 64, 32, 16])
@pytest.mark.parametrize("B,Hq,Hkv,Lq,Lkv,rounds,rows", [
    (1, 1, 1, 1, 130, 1, None), (2, 4, 2, 33, 200, 1, None), (1, 6, 3, 257, 500, 1, (5, 200)), (2, 4, 1, 100, 300, 3, None),
    (1, 8, 2, 129, 128, 4, None)])
def test_delta_formed_on_the_way_is_the_same(D, dtype, B, Hq, Hkv, Lq, Lkv, rounds, rows):
    q, k, v, do, g = _data(B, Hq, Hkv, Lq, Lkv, D, dtype, Lq + D)
    for mask in (None, _intervals(B, Lq, Lkv, g)):
        o, lse = _forward(q, k, v, mask)
        got, want = (_backward(q, k, v, o, do, lse, mask, x, rounds, rows) for x in (True, False))
        assert torch.equal(got[0], want[0])
        for a, b in zip(got[1:], want[1:]):         # (may be summed by atomics)
            torch.testing.assert_close(a.float(), b.float(), atol=1e-2 * b.float().abs().max().item(), rtol=1e-2)


@pytest.mark.gpu
@pytest.mark.parametrize("Lq,few,many", [(40, 64, 65), (300, 32, 33), (520, 21, 22), (1500, 10, 11)])
def test_tables_of_one_launch_are_those_of_two(Lq, few, many):
    """As many samples as have their tables written by one launch, and one more; no sample's gradients depend on the others."""
    q, k, v, do, g = _data(many, 2, 1, Lq, 700, 64, torch.bfloat16, Lq)
    from lv_xattn import Mask
    mask = _intervals(many, Lq, 700, g)
    mask.kv_start[:, Lq // 3:Lq // 2] = 650         # row tiles that see other token blocks than their neighbours, or nothing
    mask.kv_end[:, Lq // 3:Lq // 2] = 660
    mask.kv_end[1, Lq // 2:] = 0
    o, lse = _forward(q, k, v, mask)
    want = _backward(q, k, v, o, do, lse, mask)
    part = Mask(None, mask.kv_start[:few].contiguous(), mask.kv_end[:few].contiguous())
    got = _backward(q[:few], k[:few], v[:few], o[:few], do[:few], lse[:few * 2].contiguous(), part)
    for a, b in zip(got, want):
        torch.testing.assert_close(a.float(), b[:few].float(), atol=8e-3 * b.float().abs().max().item(), rtol=1e-2)
