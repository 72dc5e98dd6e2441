"""Rounds of the forward computed in one call: a round's parts are folded by the launch of the next one, the last round's by a
launch of their own.  Bit for bit what a call per round gives - which folds every round itself - at the edges of the
rounds, with and without an accumulator, masks, both chains of the fold, and where nothing rides along."""
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
