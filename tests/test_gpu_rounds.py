"""Rounds computed in one call.  Forward: a round's parts are folded by the launch of the next one, the last round's by a launch of
their own - bit for bit what a call per round gives, which folds every round itself - at the edges of the rounds, with and without an
accumulator, masks, both chains of the fold, and where nothing rides along.  Backward: the rows' records of all rounds are written at once, and the
slices of a round's dQ are summed by the launch of the next."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
FP32, ROUNDS = 256, 12


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.float16, 64), (torch.bfloat16, 32)])
@pytest.mark.parametrize("B,Hq,Hkv,Lq,Lkv,rounds,splits", [
    (1, 8, 2, 300, 1000, 3, 5), (2, 4, 1, 257, 700, 4, 8), (1, 4, 4, 129, 900, 2, 3), (2, 8, 2, 64, 800, 5, 12), (3, 3, 1, 1000, 300, 7, 2),
    (1, 32, 8, 2100, 500, 2, 6), (1, 4, 2, 5, 400, 4, 4), (1, 8, 2, 300, 1000, 3, 1), (1, 8, 2, 300, 1000, 3, 5 | FP32)])
@pytest.mark.parametrize("acc,masked", [(False, False), (True, False), (True, True)])
def test_rounds_in_one_call(dtype, D, B, Hq, Hkv, Lq, Lkv, rounds, splits, acc, masked, monkeypatch):
    from lv_xattn import Mask, ops
    monkeypatch.setenv("LVX_FWD_WIDE", "1")
    g = torch.Generator().manual_seed(Lq + Lkv)
    normal = lambda *shape: torch.randn(*shape, generator=g).to(dtype).to(DEV)
    # tokens outermost: rows and heads are apart; the first rows of the tensors are not the window's
    q, o_in = (normal(B, Lq + 3, Hq, D).transpose(1, 2) for _ in range(2))
    k, v = (normal(B, Lkv, Hkv, D).transpose(1, 2) for _ in range(2))
    l_in = torch.randn(B * Hq, Lq + 3, generator=g).to(DEV)
    l_in[:, ::7] = -torch.inf
    o_in[:, :, ::7] = torch.nan             # nothing has been gathered there
    mask = None
    if masked:
        row = torch.arange(Lq + 3, dtype=torch.int32).expand(B, Lq + 3)
        start = (row * 5 % (Lkv // 2)).contiguous()
        mask = Mask(None, start.to(DEV), torch.where(row % 11 == 3, start, start + Lkv // 3).int().to(DEV))
    kw = dict(acc=(o_in, l_in) if acc else None)

    def run(per_call):
        o, lse = torch.zeros_like(q), torch.zeros(B * Hq, Lq + 3, device=DEV)
        lb = -(-Lq // rounds)
        windows = [(3, Lq, splits | rounds << ROUNDS)] if not per_call else \
            [(3 + r, min(lb, Lq - r), splits) for r in range(0, Lq, lb)]
        for begin, count, n in windows:
            ws = torch.full((ops.fwd_workspace_bytes(q, k, count, n),), 0xff, dtype=torch.uint8, device=DEV)
            ops.fwd(q, k, v, o, lse, D ** -0.5, begin, count, mask, n, ws if ws.numel() else None, **kw)
        return o, lse
    a, b = run(False), run(True)
    torch.cuda.synchronize()
    assert torch.equal(a[0].isnan(), b[0].isnan()) and torch.equal(a[0].nan_to_num(), b[0].nan_to_num()) and torch.equal(a[1], b[1])
    assert a[0][:, :, 3:].nan_to_num().abs().max() > 0


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.float16, 64), (torch.bfloat16, 32)])
@pytest.mark.parametrize("B,Hq,Hkv,Lq,Lkv,rounds", [(1, 8, 2, 300, 1000, 3), (2, 4, 1, 257, 700, 4), (1, 4, 4, 129, 33, 2), (1, 8, 1, 2100, 16, 3), (1, 4, 1, 600, 500, 7), (2, 8, 2, 64, 129, 5),
                                                    (3, 3, 1, 1000, 300, 7), (1, 32, 8, 2100, 500, 2), (1, 1, 1, 5, 400, 4), (1, 40, 4, 300, 161, 2)])
@pytest.mark.parametrize("mask", [None, "lengths", "intervals"])
def test_rounds_of_the_backward_in_one_call(dtype, D, B, Hq, Hkv, Lq, Lkv, rounds, mask):
    """dQ is bit for bit what a call per round gives; dK, dV are sums of the same addends up to the order of the fp32 atomic
    ones, of which there are at most some hundred: within 2^-12 of their size."""
    from lv_xattn import Mask, ops
    g = torch.Generator().manual_seed(Lq + Lkv)
    normal = lambda *shape: torch.randn(*shape, generator=g).to(dtype).to(DEV)
    q, do = (normal(B, Lq + 3, Hq, D).transpose(1, 2) for _ in range(2))
    k, v = (normal(B, Lkv, Hkv, D).transpose(1, 2) for _ in range(2))
    kv_len = torch.tensor([Lkv, max(1, Lkv // 3), Lkv // 2][:B], dtype=torch.int32).to(DEV)
    m = None
    if mask == "lengths":
        m = Mask(kv_len)
    elif mask:
        row = torch.arange(Lq + 3, dtype=torch.int32).expand(B, Lq + 3)
        start = (row * 5 % max(1, Lkv // 2)).contiguous()
        m = Mask(kv_len, start.to(DEV), torch.where(row % 11 == 3, start, start + Lkv // 3).int().to(DEV))
    if m is not None:
        for b in range(B):
            k[b, :, kv_len[b]:], v[b, :, kv_len[b]:] = torch.nan, torch.nan
    o, lse = torch.zeros_like(q), torch.zeros(B * Hq, Lq + 3, device=DEV)
    ops.fwd(q, k, v, o, lse, D ** -0.5, 0, Lq + 3, m)
    delta = torch.zeros_like(lse)
    ops.bwd_preprocess(o, do, delta, 0, Lq + 3)
    lb = -(-Lq // rounds)

    def run(per_call):
        dq = torch.zeros_like(q)
        dk, dv = (torch.ones(B, Lkv, Hkv, D, device=DEV).transpose(1, 2) for _ in range(2))
        ws = torch.full((ops.bwd_workspace_bytes(q, k, lb, m),), 0xff, dtype=torch.uint8, device=DEV)
        for begin, count, n in [(3 + r, min(lb, Lq - r), 1) for r in range(0, Lq, lb)] if per_call else [(3, Lq, rounds)]:
            ops.bwd(q, k, v, do, lse, delta, dq, dk, dv, D ** -0.5, begin, count, m, accumulate_dkv=True, workspace=ws, rounds=n)
        return dq, dk, dv
    a, b = run(False), run(True)
    torch.cuda.synchronize()
    assert a[0][:, :, 3:].abs().max() > 0 and torch.equal(a[0], b[0])
    for x, y in zip(a[1:], b[1:]):
        assert torch.isfinite(x).all() and (x - y).abs().max() <= 2 ** -12 * y.abs().max()
