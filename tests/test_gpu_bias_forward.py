"""The forward with a dense bias at head dimensions 128 and 64: row blocks and key tiles at their edges, biases per sample and head or
shared, rows that end with the tensor, windows, key ranges, holes of -inf, with and without intervals."""
import pytest
import torch

from parity import check_lse, check_o

DEV = "cuda:0"


def _exact(q, k, v, bias, hidden):
    g = q.shape[1] // k.shape[1]
    qd, kd, vd = q.double().cpu(), k.double().cpu().repeat_interleave(g, 1), v.double().cpu().repeat_interleave(g, 1)
    s = qd @ kd.transpose(2, 3) * q.shape[-1] ** -0.5 + bias.double().cpu()
    if hidden is not None:
        s = s.masked_fill(hidden.cpu()[:, None], -float("inf"))
    return (torch.softmax(s, -1).nan_to_num(0.0) @ vd).float(), torch.logsumexp(s, -1).float()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("B,Hq,Hkv,Lq,Lkv,shared,splits,pad", [
    (1, 1, 1, 1, 1, "", 1, 0), (1, 4, 1, 63, 60, "h", 1, 0), (2, 2, 2, 65, 64, "b", 1, 4), (1, 3, 3, 64, 65, "", 1, 0),
    (2, 4, 2, 257, 130, "bh", 2, 0), (1, 8, 2, 130, 513, "h", 3, 60), (1, 2, 1, 300, 1027, "", 4, 0), (3, 4, 4, 33, 258, "b", 1, 1)])
def test_against_64_bits(D, dtype, B, Hq, Hkv, Lq, Lkv, shared, splits, pad, monkeypatch):
    from lv_xattn import Mask, ops
    monkeypatch.setenv("LVX_FWD_WIDE", "1")
    g = torch.Generator(device=DEV).manual_seed(Lq * Lkv + D)
    q, k, v = (torch.empty(B, h, n, D, dtype=dtype, device=DEV).normal_(generator=g) for h, n in ((Hq, Lq), (Hkv, Lkv), (Hkv, Lkv)))
    row = (Lkv + 3) // 4 * 4 + 4 * pad
    mem = torch.empty(1 if "b" in shared else B, 1 if "h" in shared else Hq, Lq, row, device=DEV).normal_(0.0, 2.0, generator=g)
    mem[..., Lkv:] = float("nan")                       # what is no key's is not used
    bias = mem[..., :Lkv]
    bias.masked_fill_(torch.rand(bias.shape, generator=g, device=DEV) < 0.1, -float("inf"))
    start = torch.randint(0, max(1, Lkv // 3), (B, Lq), generator=g, device=DEV, dtype=torch.int32)
    end = (start + torch.randint(1, Lkv + 1, (B, Lq), generator=g, device=DEV, dtype=torch.int32)).clamp(max=Lkv)
    if Lq > 2:
        end[-1, Lq // 2] = start[-1, Lq // 2]           # a row that sees nothing, whose bias is no number
        if "b" not in shared:
            bias[-1, :, Lq // 2] = float("nan")
    at = torch.arange(Lkv, device=DEV)
    hidden = (at < start[..., None]) | (at >= end[..., None])
    for mask, hide in ((Mask(None, start, end), hidden), (None, None)):
        full = bias.expand(B, Hq, Lq, Lkv)
        if hide is None and Lq > 2 and "b" not in shared:
            bias[-1, :, Lq // 2] = -float("inf")        # and without intervals, one that the bias hides whole
        want, want_lse = _exact(q, k, v, full, hide)
        for r0, n in ((0, Lq), (Lq // 3, Lq - Lq // 2)):
            o, lse = torch.zeros_like(q), torch.zeros(B * Hq, Lq, device=DEV)
            ws = torch.full((max(16, ops.fwd_workspace_bytes(q, k, n, splits | 256)),), 0xff, dtype=torch.uint8, device=DEV)
            ops.fwd(q, k, v, o, lse, D ** -0.5, r0, n, mask, splits | (256 if splits > 1 else 0), ws, bias)
            assert (o[:, :, :r0] == 0).all() and (o[:, :, r0 + n:] == 0).all()
            check_o(o[:, :, r0:r0 + n].cpu(), want[:, :, r0:r0 + n])
            check_lse(lse.cpu().reshape(B, Hq, Lq)[:, :, r0:r0 + n], want_lse[:, :, r0:r0 + n])


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["1", None])
def test_a_bias_that_outgrows_the_exponent(form, monkeypatch):
    """Fill values of the type's lowest, in whole rows and in part of others."""
    from lv_xattn import ops
    if form:
        monkeypatch.setenv("LVX_FWD_WIDE", form)
    g = torch.Generator(device=DEV).manual_seed(3)
    q, k, v = (torch.empty(1, 2, n, 128, dtype=torch.float16, device=DEV).normal_(generator=g) for n in (70, 200, 200))
    bias = torch.zeros(1, 1, 70, 200, device=DEV)
    bias[..., 100:] = torch.finfo(torch.float32).min
    bias[:, :, 5] = -65504.0
    bias[:, :, 6] = 1e30
    bias[:, :, 7] = -1e9
    o, lse = torch.empty_like(q), torch.empty(2, 70, device=DEV)
    ops.fwd(q, k, v, o, lse, 128 ** -0.5, bias=bias)
    want, want_lse = _exact(q, k, v, bias, None)
    keep = [i for i in range(70) if i not in (6, 7)]    # there the scores are gone in fp32: an average of V
    check_o(o[:, :, keep].cpu(), want[:, :, keep])
    for i in (6, 7):
        check_o(o[:, :, i].cpu(), v.float().mean(2).cpu())
    assert torch.allclose(lse.cpu()[:, keep], want_lse[0][:, keep], rtol=1e-6, atol=1e-3)


@pytest.mark.gpu
@pytest.mark.parametrize("row", [(1 << 22) - 4, 1 << 22])
def test_rows_of_a_bias_that_are_far_apart(row, monkeypatch):
    from lv_xattn import ops
    monkeypatch.setenv("LVX_FWD_WIDE", "1")
    g = torch.Generator(device=DEV).manual_seed(4)
    q, k, v = (torch.empty(1, 2, n, 64, dtype=torch.bfloat16, device=DEV).normal_(generator=g) for n in (70, 130, 130))
    bias = torch.empty(70 * row, device=DEV)[:69 * row + 132].as_strided((1, 1, 70, 130), (0, 0, row, 1)).normal_(generator=g)
    o, lse = torch.empty_like(q), torch.empty(2, 70, device=DEV)
    ops.fwd(q, k, v, o, lse, 0.125, bias=bias)
    want, want_lse = _exact(q, k, v, bias, None)
    check_o(o.cpu(), want)
    check_lse(lse.cpu(), want_lse[0])


def test_the_ranges_of_a_launch_with_a_bias():
    """Few rows in the plain form's many ranges, many in the wide form's few; 16-bit parts only where the plain form had them."""
    from lv_xattn.attn import auto_kv_splits
    cut = [auto_kv_splits(1, 16, 16, rows, keys, 128, True) for rows, keys in ((1, 4096), (1024, 4096), (1024, 400), (4096, 4096), (1500, 1100))]
    assert [n & 255 for n in cut[:4]] == [32, 4, 1, 1] and (cut[4] & 255 == 1 or cut[4] & 256)
