"""Masked backwards whose token blocks the device hands to work-groups: blocks cut into ranges, blocks nobody sees, whole
rounds, lists that do not divide by the XCDs, ragged last blocks, the longest lists - against the form that adds every block to fp32 accumulators as it comes."""
import pytest
import torch

DEV = "cuda:0"


def _run(q, k, v, o, do, lse, mask, accumulate):
    from lv_xattn import ops
    dq = torch.empty_like(q)
    make = torch.zeros if accumulate else torch.empty
    dk, dv = (make(k.shape[0], k.shape[2], k.shape[1], k.shape[3], dtype=torch.float32 if accumulate else q.dtype, device=DEV).transpose(1, 2)
              for _ in range(2))
    if not accumulate:
        dk.fill_(float("nan")), dv.fill_(float("nan"))
    ws = torch.full((ops.bwd_workspace_bytes(q, k, q.shape[2], mask),), 0xff, dtype=torch.uint8, device=DEV)
    ops.bwd(q, k, v, do, lse, None, dq, dk, dv, q.shape[-1] ** -0.5, mask=mask, accumulate_dkv=accumulate, workspace=ws, o=o)
    return dq, dk, dv


def _close(got, want, dtype):
    err = ((got.float() - want).norm() / want.norm()).item()
    assert torch.isfinite(got.float()).all() and err < (4e-3 if dtype == torch.bfloat16 else 1e-3), err      # one rounding of the result


@pytest.mark.gpu
@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (64, torch.float16), (32, torch.bfloat16), (16, torch.float16)])
@pytest.mark.parametrize("B,Hq,Hkv,Lq,Lkv,images,lens", [
    (1, 16, 8, 700, 70 * 128, 1, False),            # 70 equal blocks an XCD: six cut
    (2, 32, 8, 700, 37 * 128 - 60, 2, False),       # two lengths and dead blocks
    (1, 16, 8, 1100, 64 * 128, 1, True),            # whole rounds
    (2, 12, 3, 600, 99 * 128 + 1, 3, True),         # 600 blocks over 8 XCDs, of several heads and samples each
    (3, 8, 8, 200, 2800, 2, False), (2, 16, 8, 1300, 9000, 5, True), (1, 2, 2, 90, 256 * 128 * 4, 1, False)])
def test_every_block_is_summed_once(D, dtype, B, Hq, Hkv, Lq, Lkv, images, lens):
    from lv_xattn import Mask, _attn_forward
    g = torch.Generator(device=DEV).manual_seed(Lq + Lkv + D)
    q, do = (torch.empty(B, Hq, Lq, D, dtype=dtype, device=DEV).normal_(generator=g) for _ in range(2))
    k, v = (torch.empty(B, Hkv, Lkv, D, dtype=dtype, device=DEV).normal_(generator=g) for _ in range(2))
    start, end = (torch.zeros(B, Lq, dtype=torch.int32, device=DEV) for _ in range(2))
    for b in range(B):
        n = max(1, images - b)
        for i in range(n):          # the rows behind an image see it, the first few nothing, one all
            r0, r1 = Lq // 20 + (Lq - Lq // 20) * i // n, Lq // 20 + (Lq - Lq // 20) * (i + 1) // n
            start[b, r0:r1], end[b, r0:r1] = i * (Lkv // images), (i + 1) * (Lkv // images)
    start[-1, Lq // 2], end[-1, Lq // 2] = 0, Lkv
    kv_len = torch.tensor([Lkv - 150 * b - 1 for b in range(B)], dtype=torch.int32, device=DEV) if lens else None
    mask = Mask(kv_len, start, end)
    o, lse = _attn_forward(q, k, v, False, D ** -0.5, None, rounds=1, batched=True, mask=mask)[3:]
    want = _run(q, k, v, o, do, lse, mask, True)
    for _ in range(2):
        got = _run(q, k, v, o, do, lse, mask, False)
        assert torch.equal(got[0], want[0])
        _close(got[1], want[1], dtype)
        _close(got[2], want[2], dtype)
        for x, y in zip(got[1:], want[1:]):
            assert (x[y == 0] == 0).all()           # what nobody sees


@pytest.mark.gpu
@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (64, torch.float16), (32, torch.bfloat16), (16, torch.float16)])
@pytest.mark.parametrize("B,Hq,Hkv,Lq,Lkv", [
    (1, 16, 4, 540, 1346),          # every block cut alike, 6 or 5 an XCD
    (1, 64, 8, 700, 700), (1, 8, 1, 2100, 1000),        # one block an XCD and more
    (3, 12, 3, 500, 5000),          # 45 an XCD: whole rounds, the others cut
    (1, 32, 8, 1000, 6404),         # two groups of others
    (1, 8, 2, 600, 300)])           # six blocks: sums by atomics
def test_blocks_of_several_work_groups(D, dtype, B, Hq, Hkv, Lq, Lkv):
    from lv_xattn import _attn_forward
    g = torch.Generator(device=DEV).manual_seed(Lq + D)
    q, do = (torch.empty(B, Hq, Lq, D, dtype=dtype, device=DEV).normal_(generator=g) for _ in range(2))
    k, v = (torch.empty(B, Hkv, Lkv, D, dtype=dtype, device=DEV).normal_(generator=g) for _ in range(2))
    o, lse = _attn_forward(q, k, v, False, D ** -0.5, None, rounds=1, batched=True)[3:]
    want = _run(q, k, v, o, do, lse, None, True)
    got, again = (_run(q, k, v, o, do, lse, None, False) for _ in range(2))
    assert torch.equal(got[0], want[0])
    for x, y, z in zip(got[1:], want[1:], again[1:]):
        _close(x, y, dtype)
        assert B * Hkv * -(-Lkv // 128) < 8 or torch.equal(x, z)        # slices are added in one order
