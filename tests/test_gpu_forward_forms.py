"""The forward kernel's wide form (head dimensions 128 and 64) and its form for few rows (all four), at the
sizes where their tiles begin and end, against the fp32 oracle."""
import random

import pytest
import torch

from oracle import lvx_oracle as orc
from parity import check_lse, check_o

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(D, dtype, B, Hq, Hkv, Lq, Lkv, splits, mask_kind, seed):
    import lv_xattn
    from lv_xattn import _lib
    _lib.load()
    rng = random.Random(seed)
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(B, h, n, D, generator=g).to(dtype) for h, n in ((Hq, Lq), (Hkv, Lkv), (Hkv, Lkv)))
    mask, allowed, bias = None, None, None
    if mask_kind == "bias":         # every fifth key and one whole row are masked
        bias = torch.randn(B, 1, Lq, Lkv, generator=g)
        bias[..., ::5] = bias[:, :, Lq // 2] = float("-inf")
    elif mask_kind == "kv_len":
        n = torch.tensor([rng.randint(0, Lkv) for _ in range(B)], dtype=torch.int32)
        mask = lv_xattn.Mask(n)
        allowed = (torch.arange(Lkv) < n[:, None])[:, None].expand(B, Lq, Lkv)
    elif mask_kind != "none":
        # any two ends (some intervals empty, most tiles cut by some row), or whole images of 100 keys
        start = torch.randint(0, Lkv, (B, Lq), generator=g, dtype=torch.int32)
        end = torch.randint(0, Lkv + 1, (B, Lq), generator=g, dtype=torch.int32)
        if mask_kind == "images":
            start = start // 100 * 100
            end = (start + 100).clamp(max=Lkv).int()
        mask = lv_xattn.Mask(None, start, end)
        allowed = orc.interval_mask(start.long(), end.long(), Lkv)
    o_ref, l_ref = orc.attention_dense(q, k, v, D ** -0.5, bias=bias, allowed=allowed)
    bias_args = {} if bias is None else dict(bias_func=lambda b: b, local_bias_args=[bias.to(DEV)])
    _, _, _, o, lse = lv_xattn._attn_forward(q.to(DEV), k.to(DEV), v.to(DEV), False, D ** -0.5, None, rounds=1,
                                             batched=True, mask=mask, kv_splits=splits, **bias_args)
    torch.cuda.synchronize()
    check_o(o, o_ref)
    check_lse(lse, l_ref)


# key counts around one, two and three tiles of 64; row counts around one and two work-groups (64 rows
# of four heads, 128 of two, 256 of one)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("Hq,Hkv,Lq,Lkv,splits,mask", [
    (4, 1, 1, 1, 1, "none"), (4, 1, 64, 64, 1, "none"), (4, 1, 65, 65, 1, "none"), (4, 1, 63, 128, 1, "none"),
    (8, 2, 128, 129, 1, "kv_len"), (2, 2, 257, 192, 1, "none"), (4, 2, 129, 193, 1, "intervals"),
    (4, 1, 64, 257, 2, "intervals"), (8, 1, 100, 700, 3, "images"), (3, 1, 70, 640, 1, "images"),
    (4, 1, 10, 4300, 64, "none")])
def test_wide_form(D, dtype, Hq, Hkv, Lq, Lkv, splits, mask, monkeypatch):
    monkeypatch.setenv("LVX_FWD_WIDE", "1")
    _check(D, dtype, 2, Hq, Hkv, Lq, Lkv, splits, mask, Lq * 1000 + Lkv)


# key counts around one piece of 32, one round of the four waves (128) and two (256); columns (rows x heads
# of the group) around one tile of 32
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [128, 64, 32, 16])
@pytest.mark.parametrize("Hq,Hkv,Lq,Lkv,splits,mask", [
    (4, 1, 1, 1, 1, "none"), (4, 1, 8, 32, 1, "none"), (4, 1, 9, 33, 1, "none"), (1, 1, 31, 128, 1, "none"),
    (8, 2, 1, 129, 1, "kv_len"), (3, 1, 11, 257, 1, "none"), (8, 1, 4, 511, 2, "intervals"),
    (2, 1, 128, 300, 1, "images"), (4, 2, 3, 2500, 64, "none"), (4, 4, 5, 700, 5, "images")])
def test_few_rows_form(D, dtype, Hq, Hkv, Lq, Lkv, splits, mask, monkeypatch):
    monkeypatch.setenv("LVX_FWD_WIDE", "2")
    _check(D, dtype, 2, Hq, Hkv, Lq, Lkv, splits, mask, Lq * 1000 + Lkv + 1)


# with a dense bias, whose values are requested a tile ahead: one tile and less, two, the last of them partial, key
# ranges that begin inside the bias, every grouping of heads and rows into a work-group
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [128, 64, 32, 16])
@pytest.mark.parametrize("Hq,Hkv,Lq,Lkv,splits", [
    (1, 1, 1, 1, 1), (4, 1, 33, 63, 1), (4, 4, 129, 64, 1), (2, 1, 65, 65, 1), (4, 2, 31, 130, 2), (3, 1, 40, 257, 1), (8, 1, 32, 1000, 5)])
def test_form_with_a_bias(D, dtype, Hq, Hkv, Lq, Lkv, splits):
    _check(D, dtype, 2, Hq, Hkv, Lq, Lkv, splits, "bias", Lq * 1000 + Lkv + 2)


# nothing in a forward depends on the order in which anything arrives
@pytest.mark.parametrize("form", ["1", "2"])
@pytest.mark.parametrize("D", [128, 64, 32])
def test_every_form_repeats_itself(D, form, monkeypatch):
    import lv_xattn
    monkeypatch.setenv("LVX_FWD_WIDE", form)
    g = torch.Generator(device=DEV).manual_seed(D)
    q, k, v = (torch.empty(2, h, n, D, device=DEV, dtype=torch.bfloat16).normal_(generator=g) for h, n in ((32, 7), (8, 3000), (8, 3000)))
    first = None
    for _ in range(20):
        _, _, _, o, lse = lv_xattn._attn_forward(q, k, v, False, D ** -0.5, None, rounds=1, batched=True)
        first = first or (o, lse)
        assert torch.equal(o, first[0]) and torch.equal(lse, first[1])


# the parts of key splits in fp32 (LVX_SPLITS_FP32), at the edges of every form's tiles
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [128, 64, 32, 16])
@pytest.mark.parametrize("form", ["1", "2"])
@pytest.mark.parametrize("Hq,Hkv,Lq,Lkv,splits,mask", [
    (4, 1, 1, 65, 2, "none"), (4, 1, 63, 129, 3, "intervals"), (8, 2, 33, 300, 5, "kv_len"), (2, 2, 65, 700, 9, "images"),
    (4, 2, 3, 2500, 64, "none"), (4, 2, 65, 129, 2, "bias"), (8, 2, 3, 700, 9, "bias")])
def test_parts_in_fp32(D, dtype, form, Hq, Hkv, Lq, Lkv, splits, mask, monkeypatch):
    monkeypatch.setenv("LVX_FWD_WIDE", form)
    _check(D, dtype, 2, Hq, Hkv, Lq, Lkv, splits | 256, mask, Lq * 1000 + Lkv + 2)


# few rows, a short range, and 528 work-groups of 32-row waves (a last round that the splits even out).  A part in
# 16 bits would add a rounding of the size of the result's own, sqrt(2) in quadrature less what P's rounding
# adds to both: 1.2 measured; 1.05 leaves room for the sample (at least 25600 elements, 1 % of a norm).
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Lq,Lkv", [(25, 929), (256, 929), (2100, 6404)])
def test_splits_chosen_by_the_library_keep_the_precision_of_a_whole_launch(Lq, Lkv, dtype):
    import lv_xattn
    from lv_xattn.attn import auto_kv_splits
    B, Hq, Hkv, D = 1, 32, 8, 128
    assert auto_kv_splits(B, Hq, Hkv, Lq, Lkv) & 255 > 1
    g = torch.Generator(device=DEV).manual_seed(Lq)
    q, k, v = (torch.empty(B, h, n, D, device=DEV, dtype=dtype).normal_(generator=g) for h, n in ((Hq, Lq), (Hkv, Lkv), (Hkv, Lkv)))
    error = []
    for splits in (None, 1):
        o = lv_xattn._attn_forward(q, k, v, False, D ** -0.5, None, rounds=1, batched=True, kv_splits=splits)[3]
        diff = ref = 0.0
        for h in range(0, Hq, 4):
            exact = torch.softmax(q[0, h].double() @ k[0, h // 4].double().T.contiguous() * D ** -0.5, -1) @ v[0, h // 4].double()
            diff += (o[0, h].double() - exact).square().sum().item()
            ref += exact.square().sum().item()
        error.append((diff / ref) ** 0.5)
    assert error[0] < 1.05 * error[1], error


# Rows with an empty interval (padding, whose q may hold anything) among rows that see keys: zeros and -inf, exactly
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("form,D", [("1", 128), ("1", 64), ("1", 32), ("1", 16), ("2", 128), ("2", 64), ("2", 32), ("2", 16)])
@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("junk", [float("nan"), float("inf")])
def test_a_row_that_sees_nothing_is_zero_whatever_its_q(form, D, dtype, splits, junk, monkeypatch):
    import lv_xattn
    monkeypatch.setenv("LVX_FWD_WIDE", form)
    B, Hq, Hkv, Lq, Lkv = 2, 4, 2, 40, 300
    g = torch.Generator().manual_seed(D)
    q, k, v = (torch.randn(B, h, n, D, generator=g).to(dtype) for h, n in ((Hq, Lq), (Hkv, Lkv), (Hkv, Lkv)))
    start = torch.randint(0, Lkv - 1, (B, Lq), generator=g, dtype=torch.int32)
    end = torch.randint(1, Lkv + 1, (B, Lq), generator=g, dtype=torch.int32)
    end = torch.maximum(end, start + 1)
    dead = torch.arange(Lq)[None] % 3 == torch.tensor([[0], [1]])
    end[dead] = start[dead] - torch.arange(Lq).expand(B, Lq)[dead].int() % 2        # [s, s) and [s, s - 1)
    o_ref, l_ref = orc.attention_dense(q, k, v, D ** -0.5, allowed=orc.interval_mask(start.long(), end.long(), Lkv))
    q.transpose(1, 2)[dead] = junk
    _, _, _, o, lse = lv_xattn._attn_forward(q.to(DEV), k.to(DEV), v.to(DEV), False, D ** -0.5, None, rounds=1, batched=True,
                                             mask=lv_xattn.Mask(None, start, end), kv_splits=splits)
    check_o(o, o_ref)
    check_lse(lse, l_ref)
    assert not o.cpu().transpose(1, 2)[dead].any()


# A NaN among a row's scores gives a row of NaN, whether its keys are cut into ranges (with the range that holds it
# in any place) or not; the other rows, and the heads it is not in, stay as they are.
@pytest.mark.parametrize("form,D,kind", [("1", 128, "none"), ("1", 64, "images"), ("1", 32, "none"), ("1", 128, "bias"),
                                         ("2", 128, "none"), ("2", 64, "images"), ("2", 16, "none")])
@pytest.mark.parametrize("splits", [1, 3, 3 | 256, 12, 12 | 256])
@pytest.mark.parametrize("key", [0, 130, 699])
def test_a_nan_is_not_lost_between_key_splits(form, D, kind, splits, key, monkeypatch):
    import lv_xattn
    monkeypatch.setenv("LVX_FWD_WIDE", form)
    B, Hq, Hkv, Lq, Lkv = 1, 4, 2, 40, 700
    g = torch.Generator().manual_seed(D)
    q, k, v = (torch.randn(B, h, n, D, generator=g).bfloat16() for h, n in ((Hq, Lq), (Hkv, Lkv), (Hkv, Lkv)))
    start, end = torch.zeros(B, Lq, dtype=torch.int32), torch.full((B, Lq), Lkv, dtype=torch.int32)
    if kind == "images":
        start[0] = torch.arange(Lq) % 7 * 100
        end = start + 100
    bias = torch.randn(B, 1, Lq, Lkv, generator=g)
    mask = lv_xattn.Mask(None, start, end) if kind == "images" else None
    bias_args = dict(bias_func=lambda b: b, local_bias_args=[bias.to(DEV)]) if kind == "bias" else {}
    o_ref, l_ref = orc.attention_dense(q, k, v, D ** -0.5, bias=bias if kind == "bias" else None,
                                       allowed=orc.interval_mask(start.long(), end.long(), Lkv))
    k[0, 1, key] = q[0, 0, 7] = float("nan")
    nan = torch.zeros(B, Hq, Lq, dtype=torch.bool)
    nan[0, 2:] = (start[0] <= key) & (key < end[0])
    nan[0, 0, 7] = True
    o = lv_xattn._attn_forward(q.to(DEV), k.to(DEV), v.to(DEV), False, D ** -0.5, None, rounds=1, batched=True, mask=mask,
                               kv_splits=splits, **bias_args)[3].cpu()
    assert torch.equal(o.isnan().all(-1), nan) and torch.equal(o.isnan().any(-1), nan)
    check_o(o[~nan], o_ref[~nan])


# rows of O further apart than 32 bits of elements reach over the rows that one store instruction covers (eight with
# heads of 64, four with heads of 128): 8.6 GB, of which only the rows are touched
@pytest.mark.parametrize("D,Lq", [(64, 8), (128, 4)])
def test_wide_form_with_rows_far_apart(D, Lq, monkeypatch):
    from lv_xattn import ops
    monkeypatch.setenv("LVX_FWD_WIDE", "1")
    g = torch.Generator(device=DEV).manual_seed(D)
    q, k, v = (torch.empty(1, 4, n, D, device=DEV, dtype=torch.bfloat16).normal_(generator=g) for n in (Lq, 100, 100))
    stride = (2 ** 32 // (Lq - 1) + 4 * D + 8) // 8 * 8
    assert (Lq - 1) * stride > 2 ** 32
    far = torch.empty((Lq - 1) * stride + 4 * D, device=DEV, dtype=torch.bfloat16).as_strided((1, 4, Lq, D), (0, D, stride, 1))
    near, lse = torch.empty_like(q), torch.empty(4, Lq, device=DEV)
    for o in (near, far):
        ops.fwd(q, k[:, :1], v[:, :1], o, lse, D ** -0.5)
    torch.cuda.synchronize()
    assert torch.equal(near, far)
