"""Launches for few rows that fold their own parts (up to four columns per kv head, fp32 parts): numbers of parts around those a
wave loads at once, one to five columns, empty ranges and rows, whatever O holds before, replays of a graph."""
import pytest
import torch

import rules
from parity import check_lse, check_o

DEV = "cuda:0"


def test_the_rule_ends_at_a_column_a_wave(tmp_path):
    asked = [(1, 1), (2, 1), (64, 4), (2, 5), (64, 32)]
    assert rules.ask(tmp_path, "lvx_fold_rule.hpp", "parts cols", "lvx::fold_inside(parts, cols)", asked) == [0, 1, 1, 0, 0]


def _forward(q, k, v, splits, mask=None, o=None):
    from lv_xattn import ops
    B, Hq, Lq, D = q.shape
    o = torch.empty_like(q) if o is None else o
    lse = torch.empty(B * Hq, Lq, dtype=torch.float32, device=DEV)
    ws = torch.full((ops.fwd_workspace_bytes(q, k, Lq, splits),), 0xff, dtype=torch.uint8, device=DEV)
    ops.fwd(q, k, v, o, lse, D ** -0.5, 0, Lq, mask, splits, ws)
    return o, lse


def _exact(q, k, v, hidden=None):
    g = q.shape[1] // k.shape[1]
    kf, vf = (t.double().repeat_interleave(g, 1) for t in (k, v))
    s = (q.double()[:, :, :, None] * kf[:, :, None]).sum(-1) * q.shape[-1] ** -0.5
    if hidden is not None:
        s = s.masked_fill(hidden[:, None], -float("inf"))
    p = torch.softmax(s, -1).nan_to_num(0.0)
    return (p[..., None] * vf[:, :, None]).sum(3).float(), torch.logsumexp(s, -1).float()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [128, 64, 32, 16])
@pytest.mark.parametrize("B,Hq,Hkv,Lq,Lkv,parts", [
    (1, 1, 1, 1, 64, 2), (3, 4, 1, 1, 500, 15), (2, 6, 3, 2, 544, 17), (1, 8, 2, 1, 1100, 33), (2, 3, 3, 3, 2048, 64), (1, 5, 1, 1, 600, 8)])
def test_against_64_bits(D, dtype, B, Hq, Hkv, Lq, Lkv, parts, monkeypatch):
    from lv_xattn import Mask
    monkeypatch.setenv("LVX_FWD_WIDE", "2")
    g = torch.Generator(device=DEV).manual_seed(Lkv + D)
    q, k, v = (torch.empty(B, h, n, D, dtype=dtype, device=DEV).normal_(generator=g) for h, n in ((Hq, Lq), (Hkv, Lkv), (Hkv, Lkv)))
    start = torch.randint(0, Lkv // 2, (B, Lq), generator=g, device=DEV, dtype=torch.int32)
    end = start + torch.randint(1, Lkv // 2, (B, Lq), generator=g, device=DEV, dtype=torch.int32)
    end[-1, -1] = start[-1, -1]                     # a row that sees nothing
    at = torch.arange(Lkv, device=DEV)
    hidden = (at < start[..., None]) | (at >= end[..., None])
    for mask, hide in ((None, None), (Mask(None, start, end), hidden)):
        o = torch.empty(B, Lq, Hq, D, dtype=dtype, device=DEV).fill_(float("nan")).transpose(1, 2)      # tokens outermost
        got, lse = _forward(q, k, v, parts | 256, mask, o)
        again, lse2 = _forward(q, k, v, parts | 256, mask)          # nothing depends on which work-group was the last
        assert torch.equal(got, again) and torch.equal(lse, lse2)
        want, want_lse = _exact(q, k, v, hide)
        check_o(got.cpu(), want.cpu())
        check_lse(lse.cpu().reshape(B, Hq, Lq), want_lse.cpu())
        if hide is not None:
            assert (got[-1, :, -1] == 0).all()


@pytest.mark.gpu
def test_a_part_that_holds_nan_makes_the_row_nan(monkeypatch):
    monkeypatch.setenv("LVX_FWD_WIDE", "2")
    q, k, v = (torch.ones(1, h, n, 64, dtype=torch.bfloat16, device=DEV) for h, n in ((4, 1), (2, 700), (2, 700)))
    k[0, 1, 450] = float("nan")
    o, lse = _forward(q, k, v, 9 | 256)
    assert (o[0, :2] == 1).all() and o[0, 2:].isnan().all() and lse[:2].isfinite().all()


@pytest.mark.gpu
def test_an_output_in_the_place_of_an_input(monkeypatch):
    """What a launch that counts in its output may not do."""
    monkeypatch.setenv("LVX_FWD_WIDE", "2")
    g = torch.Generator(device=DEV).manual_seed(1)
    q, k, v = (torch.empty(2, h, n, 128, dtype=torch.bfloat16, device=DEV).normal_(generator=g) for h, n in ((4, 1), (1, 900), (1, 900)))
    want, want_lse = _forward(q, k, v, 7)           # 16-bit parts: a fold of its own
    for _ in range(3):
        x = q.clone()
        o, lse = _forward(x, k, v, 7 | 256, o=x)
        check_o(o.cpu(), want.float().cpu())
        check_lse(lse.cpu(), want_lse.cpu())


@pytest.mark.gpu
def test_a_replayed_graph_counts_as_the_first_launch_did():
    import lv_xattn
    g = torch.Generator(device=DEV).manual_seed(2)
    q, k, v = (torch.empty(1, h, n, 128, dtype=torch.bfloat16, device=DEV).normal_(generator=g) for h, n in ((32, 1), (8, 6404), (8, 6404)))

    def run():
        return lv_xattn._attn_forward(q, k, v, False, 128 ** -0.5, None, rounds=1, batched=True)[3:]
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = run()
    for i in range(4):
        q.normal_(generator=g)
        want = [x.clone() for x in run()]
        if i == 2:
            outs[0].fill_(7.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(outs, want))
