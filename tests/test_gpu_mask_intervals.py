"""lvx_bias_hull, and lvx_mask_intervals: an additive mask as transformers builds it against the intervals it was made from, at
row lengths and alignments where the 8-byte words of a row begin before it or end behind it, and on
masks that are more than intervals."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,Lq,Lkv,offset", [(1, 1, 1, 0), (2, 3, 7, 0), (3, 4, 1601, 1), (2, 30, 333, 3), (1, 2, 4096, 2),
                                              (1, 3, 256, 3), (2, 2, 1025, 1), (1, 2, 4099, 0)])
def test_mask_intervals(dtype, B, Lq, Lkv, offset):
    from lv_xattn import ops
    g = torch.Generator().manual_seed(Lkv)
    neg = torch.finfo(dtype).min
    start = torch.randint(0, Lkv, (B, Lq), generator=g)
    end = (start + 1 + torch.randint(0, Lkv, (B, Lq), generator=g)).clamp(max=Lkv)
    keys = torch.arange(Lkv)
    visible = (keys >= start[..., None]) & (keys < end[..., None])
    memory = torch.zeros(B * Lq * Lkv + 8, dtype=dtype, device=DEV)
    mask = memory[offset:offset + B * Lq * Lkv].view(B, 1, Lq, Lkv)
    mask.masked_fill_(~visible[:, None].to(DEV), neg)
    got = ops.mask_intervals(mask)
    assert torch.equal(got.kv_start.cpu(), start.int()) and torch.equal(got.kv_end.cpu(), end.int())
    memory[:offset] = 1.0           # what lies before the first row and behind the last is no part of the mask
    memory[offset + B * Lq * Lkv:] = 1.0
    assert ops.mask_intervals(mask) is not None
    finite = mask.clone()
    finite[-1, 0, -1, int(start[-1, -1])] = 0.5
    nothing = mask.clone()
    nothing[0, 0, 0] = neg
    assert ops.mask_intervals(finite) is None and ops.mask_intervals(nothing) is None
    if Lkv > 2:
        gap = torch.zeros_like(mask)
        gap[0, 0, 0, Lkv // 2] = float("-inf")
        assert ops.mask_intervals(gap) is None


# a wave to a row with one, two and four loads in flight and a work-group to a row, at the edges of their ranges
# of keys and rows; samples and heads that share the bias or do not
@pytest.mark.parametrize("B,nb,H,nh,Lq,Lkv", [
    (1, 1, 2, 1, 1, 1), (2, 2, 2, 2, 5, 255), (3, 1, 2, 1, 2, 256), (1, 1, 2, 2, 9, 257), (2, 2, 2, 1, 3, 512), (1, 1, 3, 3, 6, 513),
    (1, 1, 2, 1, 7, 1024), (1, 1, 2, 2, 257, 1025), (2, 2, 1, 1, 128, 1025), (2, 1, 1, 1, 129, 1031), (1, 1, 2, 2, 3, 4099), (3, 3, 1, 1, 342, 4100)])
def test_hull_of_a_dense_bias(B, nb, H, nh, Lq, Lkv):
    from lv_xattn import ops
    g = torch.Generator().manual_seed(Lkv)
    bias = torch.full((nb, nh, Lq, Lkv + -Lkv % 4), -torch.inf)
    bias[..., Lkv:] = 1.0                                               # is no part of it
    for _ in range(3):                                                  # up to three finite entries per row and head
        at = torch.randint(0, Lkv, (nb, nh, Lq, 1), generator=g)
        bias.scatter_(-1, at, torch.randn(nb, nh, Lq, 1, generator=g))
    bias[0, :, 0, :Lkv] = -torch.inf                                    # an empty row
    if Lq > 1:
        bias[-1, -1, -1, 0] = bias[-1, -1, -1, Lkv - 1] = 0.0           # a whole one
    seen = (bias[..., :Lkv] > -torch.inf).any(1).expand(B, Lq, Lkv)
    start, end = seen.int().argmax(-1), Lkv - seen.int().flip(-1).argmax(-1)
    none = ~seen.any(-1)
    start[none], end[none] = 0, 0
    q, k = torch.zeros(B, H, Lq, 16, device=DEV, dtype=torch.float16), torch.zeros(B, H, Lkv, 16, device=DEV, dtype=torch.float16)
    got = ops.bias_hull(q, k, bias.to(DEV)[..., :Lkv])
    assert torch.equal(got.kv_start.cpu(), start.int()) and torch.equal(got.kv_end.cpu(), end.int())


class _Layer(torch.nn.Module):
    k_norm = None
    is_causal = False


def _attend(q, k, v, mask):
    from lv_xattn import hf_mllama
    hf_mllama.clear_mask_cache()
    return hf_mllama.lv_xattn_attention_forward(_Layer(), q, k, v, mask)[0]


def test_masks_of_another_form_take_the_general_path():
    """A mask shared by the batch and one in host memory give what the mask written out on the GPU gives;
    one with fewer keys than there are is refused as it is without intervals."""
    torch.manual_seed(0)
    q, k, v = (torch.randn(2, h, n, 64, device=DEV, dtype=torch.bfloat16) for h, n in ((8, 5), (2, 333), (2, 333)))
    mask = torch.zeros(1, 1, 5, 333, device=DEV, dtype=torch.bfloat16)
    mask[..., 100:] = torch.finfo(torch.bfloat16).min
    want = _attend(q, k, v, mask.expand(2, 1, 5, 333).contiguous())
    for other in (mask, mask.cpu()):
        torch.testing.assert_close(_attend(q, k, v, other), want, rtol=2.0 ** -7, atol=2.0 ** -7)
    with pytest.raises(ValueError):
        _attend(q, k, v, mask.expand(2, 1, 5, 333)[..., :200].contiguous())


def test_a_mask_first_seen_under_capture():
    """In inference mode a mask has no version by which an answer could be kept: a captured call takes the path
    that asks nothing of the host, and every replay reads the mask as it is then."""
    torch.manual_seed(1)
    with torch.inference_mode():
        q, k, v = (torch.randn(1, h, n, 64, device=DEV, dtype=torch.bfloat16) for h, n in ((8, 5), (2, 333), (2, 333)))
        mask = torch.zeros(1, 1, 5, 333, device=DEV, dtype=torch.bfloat16)
        _attend(q, k, v, mask)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = _attend(q, k, v, mask)
        for visible in (333, 100, 7):
            mask.zero_()
            mask[..., visible:] = torch.finfo(torch.bfloat16).min
            graph.replay()
            torch.cuda.synchronize()
            torch.testing.assert_close(out, _attend(q, k, v, mask), rtol=2.0 ** -7, atol=2.0 ** -7)


def _capture(stream, q, k, v, mask):
    from lv_xattn import hf_mllama
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = hf_mllama.lv_xattn_attention_forward(_Layer(), q, k, v, mask)[0]
    return graph, out


def _replays_read_the_mask(graph, out, q, k, v, mask):
    """Every replay sees the mask as it is then, with eager work, other masks and synchronizations in between."""
    for visible in (mask.shape[-1], 100, 7, mask.shape[-1] - 1):
        new = torch.zeros_like(mask)
        new[..., visible:] = torch.finfo(mask.dtype).min
        want = _attend(q, k, v, new)
        mask.copy_(new)
        graph.replay()
        torch.cuda.synchronize()
        torch.testing.assert_close(out, want, rtol=2.0 ** -7, atol=2.0 ** -7)


# 20000 keys: long enough for torch to share a reduction over a row among several blocks
@pytest.mark.parametrize("keys", [333, 20000])
def test_an_ordinary_mask_under_capture_after_an_eager_warm_up(keys):
    """As generation with a static mask buffer has it: eager calls on the default stream, then a capture on
    torch.cuda.graph's own, nothing cleared in between."""
    torch.manual_seed(2)
    with torch.no_grad():
        q, k, v = (torch.randn(1, h, n, 64, device=DEV, dtype=torch.bfloat16) for h, n in ((8, 1), (2, keys), (2, keys)))
        mask = torch.zeros(1, 1, 1, keys, device=DEV, dtype=torch.bfloat16)
        mask[..., keys // 2:] = torch.finfo(torch.bfloat16).min
        _attend(q, k, v, mask)
        torch.cuda.synchronize()
        graph, out = _capture(None, q, k, v, mask)
        _replays_read_the_mask(graph, out, q, k, v, mask)


@pytest.mark.parametrize("plain", [True, False])
def test_a_capture_on_the_stream_of_the_warm_up(plain):
    """What the warm-up kept for this very stream - the intervals, or the converted mask of one that is more than
    intervals - is not what a replay may use once the mask was written to."""
    torch.manual_seed(3)
    side = torch.cuda.Stream()
    with torch.no_grad():
        q, k, v = (torch.randn(1, h, n, 64, device=DEV, dtype=torch.bfloat16) for h, n in ((8, 3), (2, 400), (2, 400)))
        mask = torch.zeros(1, 1, 3, 400, device=DEV, dtype=torch.bfloat16)
        mask[..., 50:] = torch.finfo(torch.bfloat16).min
        if not plain:
            mask[..., 10] = -1.0
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            _attend(q, k, v, mask)
        torch.cuda.synchronize()
        graph, out = _capture(side, q, k, v, mask)
        _replays_read_the_mask(graph, out, q, k, v, mask)
