"""The Hugging Face attention function's host side, with the kernels replaced by stand-ins: what it
refuses, what it hands to autograd."""
import pytest
import torch
from torch.autograd import forward_ad

from lv_xattn import attn, autograd, hf_mllama, ops


class _Layer(torch.nn.Module):
    k_norm = None
    is_causal = False


@pytest.fixture
def no_kernels(monkeypatch):
    def forward(q, k, v, causal, scale, mode, *args, _token_major=False, **kw):
        B, H, L, D = q.shape
        o = torch.zeros(B, L, H, D, dtype=q.dtype).transpose(1, 2) if _token_major else torch.zeros(B, H, L, D, dtype=q.dtype)
        return q, k, v, o, torch.zeros(B * H, L)

    def backward(do, q, k, v, *args, **kw):
        return torch.ones_like(q), torch.ones_like(k), torch.ones_like(v)

    for module in (hf_mllama, autograd):
        monkeypatch.setattr(module, "_attn_forward", forward)
    monkeypatch.setattr(autograd, "_attn_backward", backward)
    monkeypatch.setattr(hf_mllama, "_require_supported", lambda *a: None)


def _qkv():
    return tuple(torch.randn(1, h, n, 64).bfloat16() for h, n in ((8, 5), (2, 33), (2, 33)))


@pytest.mark.parametrize("which", [0, 1, 2])
@pytest.mark.parametrize("grad", [True, False])
def test_a_forward_mode_tangent_is_refused(no_kernels, which, grad):
    """The kernels have no forward-mode derivative: an input with a tangent raises, as an autograd function
    without a jvp does, instead of giving an output that reads as derivative zero."""
    with torch.set_grad_enabled(grad), forward_ad.dual_level():
        qkv = list(_qkv())
        assert hf_mllama.lv_xattn_attention_forward(_Layer(), *qkv, None)[0].shape == (1, 5, 8, 64)
        qkv[which] = forward_ad.make_dual(qkv[which], torch.ones_like(qkv[which]))
        with pytest.raises(NotImplementedError, match="jvp"):
            hf_mllama.lv_xattn_attention_forward(_Layer(), *qkv, None)


class _Net(_Layer):
    def forward(self, q, k, v, mask=None):
        return hf_mllama.lv_xattn_attention_forward(self, q, k, v, mask)[0]


@pytest.mark.filterwarnings("ignore")       # the tracer's, about the stand-in
def test_a_traced_call_computes(monkeypatch):
    """torch.jit.trace without gradients: what it records runs the kernels on the inputs of each later call.  The
    kernels write where the tracer does not look, so a trace without the autograd function would return memory that
    nothing has written.  A mask, which the function takes in a list, is refused by the tracer, where the intervals
    of the mask it saw would be a constant to it."""
    def forward(q, k, v, causal, scale, mode, bias_func=None, local=(), *args, mask=None, _token_major=False, **kw):
        assert mask is None
        bias_func is None or bias_func(*local)
        o = torch.empty(q.shape)
        o.detach().numpy()[...] = 5 * q.detach().numpy()
        return q, k, v, o, torch.zeros(q.shape[0] * q.shape[1], q.shape[2])

    for module in (hf_mllama, autograd):
        monkeypatch.setattr(module, "_attn_forward", forward)
    monkeypatch.setattr(hf_mllama, "_require_supported", lambda *a: None)
    monkeypatch.setattr(ops, "mask_intervals", lambda mask: ops.Mask())
    hf_mllama.clear_mask_cache()
    with torch.no_grad():
        traced = torch.jit.trace(_Net(), tuple(t.float() for t in _qkv()), check_trace=False)
        q, k, v = (t.float() for t in _qkv())
        assert torch.equal(traced(q, k, v), 5 * q.transpose(1, 2))
        with pytest.raises(RuntimeError):
            torch.jit.trace(_Net(), (q, k, v, _mask(20)), check_trace=False)
    hf_mllama.clear_mask_cache()


class _Gpu:
    """Stands in for the current stream: its number, and whether it is capturing."""

    def __init__(self, monkeypatch):
        self.stream, self.capturing, self.waits = 1, False, []
        monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: self.capturing)
        monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: self)

        def intervals(mask):
            assert not self.capturing, "a host read under capture"
            self.waits.append("mask_intervals")
            visible = mask[:, 0] > -30000
            first = visible.int().argmax(-1)
            return ops.Mask(None, first.int(), (first + visible.sum(-1)).int())

        def is_interval(*a):
            assert not self.capturing, "a host read under capture"
            self.waits.append("bias_is_interval")
            return True

        monkeypatch.setattr(ops, "mask_intervals", intervals)
        monkeypatch.setattr(ops, "bias_is_interval", is_interval)
        monkeypatch.setattr(ops, "bias_hull", lambda *a: ops.Mask())

    @property
    def cuda_stream(self):
        return self.stream


@pytest.fixture
def gpu(monkeypatch):
    hf_mllama.clear_mask_cache()
    yield _Gpu(monkeypatch)
    hf_mllama.clear_mask_cache()


@pytest.fixture
def seen(monkeypatch):
    """What the kernels are given of a call's mask: the intervals, or the dense bias."""
    calls = []

    def forward(q, k, v, causal, scale, mode, bias_func=None, local=(), remote=(), *args, mask=None, **kw):
        bias = attn._dense_bias(bias_func, local, remote, q.shape[0], q.shape[1], q.shape[2], k.shape[2], q.device)
        if mask is None and bias is not None:
            bias, mask = attn._bias_and_hull(bias, q, k)
        calls.append((mask, bias))
        return q, k, v, torch.zeros_like(q), torch.zeros(q.shape[0] * q.shape[1], q.shape[2])

    for module in (hf_mllama, autograd):
        monkeypatch.setattr(module, "_attn_forward", forward)
    monkeypatch.setattr(hf_mllama, "_require_supported", lambda *a: None)
    return calls


def _mask(visible):
    mask = torch.zeros(1, 1, 5, 33, dtype=torch.bfloat16)
    mask[..., visible:] = torch.finfo(torch.bfloat16).min
    return mask


def test_a_captured_call_reads_nothing_back(gpu, seen):
    """A warm-up on one stream and a capture on another, as torch.cuda.graph has it: the captured calls ask
    nothing of the host, and nothing a capture recorded (but did not compute) is kept for a later call."""
    q, k, v = _qkv()
    mask = _mask(20)
    with torch.no_grad():
        hf_mllama.lv_xattn_attention_forward(_Layer(), q, k, v, mask)
        gpu.stream, gpu.capturing = 2, True
        for _ in range(2):
            hf_mllama.lv_xattn_attention_forward(_Layer(), q, k, v, mask)
        gpu.capturing = False
        recorded = [bias for _, bias in seen[1:]]
        assert all(b is not None for b in recorded)
        assert all(b is not hf_mllama._mask_bias(mask) and not hasattr(b, "lvx_hull") for b in recorded)


@pytest.mark.parametrize("keys", [1, 1023, 1024, 2047, 2048, 2049, 5000])
def test_a_row_that_sees_one_key_anywhere(keys):
    visible = torch.zeros(3, 1, keys, keys, dtype=torch.bool) if keys < 10 else torch.zeros(1, 1, 4, keys, dtype=torch.bool)
    for row, key in enumerate((0, keys // 2, keys - 1)[:visible.shape[2]]):
        visible[0, 0, row, key] = True
    assert torch.equal(hf_mllama._sees_a_key(visible), visible.any(-1, keepdim=True))


def test_a_capture_uses_no_answer_that_was_kept(gpu, seen):
    """On the very stream of the warm-up: the captured calls convert the mask in the graph, whether the intervals or
    the converted mask had been kept, so that a replay reads the mask as it is then."""
    q, k, v = _qkv()
    with torch.no_grad():
        for mask in (_mask(20), _mask(20).masked_fill(torch.arange(33) == 3, -1.0)):     # an interval mask, and another
            hf_mllama.lv_xattn_attention_forward(_Layer(), q, k, v, mask)
            kept = hf_mllama._mask_bias(mask)
            gpu.capturing = True
            hf_mllama.lv_xattn_attention_forward(_Layer(), q, k, v, mask)
            gpu.capturing = False
            assert seen[-1][1] is not None and seen[-1][1] is not kept


def test_layers_in_inference_mode_wait_for_nothing(gpu, seen):
    """A mask without a version counter: nothing can be kept for it, so nothing that has to come back to the host is
    asked in any of the layers; with a version, the first layer asks and the others find the answer."""
    with torch.inference_mode():
        q, k, v = _qkv()
        mask = _mask(20)
        for _ in range(4):
            hf_mllama.lv_xattn_attention_forward(_Layer(), q, k, v, mask)
    assert gpu.waits == [] and all(bias is not None for _, bias in seen)
    with torch.no_grad():
        q, k, v = _qkv()
        mask = _mask(20)
        for _ in range(4):
            hf_mllama.lv_xattn_attention_forward(_Layer(), q, k, v, mask)
    assert gpu.waits == ["mask_intervals"]


def test_the_result_of_a_recorded_call_may_be_written_to(no_kernels):
    """A caller may scale or mask the attention's output in place before it is projected: what backward needs is
    not that memory."""
    q, k, v = (t.requires_grad_() for t in _qkv())
    out = hf_mllama.lv_xattn_attention_forward(_Layer(), q, k, v, None)[0]
    assert out.is_contiguous() and out.shape == (1, 5, 8, 64)
    out.mul_(0.5)
    out.float().sum().backward()
    assert all(t.grad is not None for t in (q, k, v))


def test_a_projection_without_a_norm_inside_run_function(monkeypatch):
    """run_function may project a part that needs no gradient - here q, from frozen weights on detached states -
    without a norm, in both of its runs."""
    calls = []

    def q_proj(x, w, heads, w_in_major=True, norm=None, eps=1e-5, for_backward=False):
        assert norm is not None or not for_backward        # ops.q_proj refuses that
        calls.append(for_backward)
        q = (x @ w).view(x.shape[0], x.shape[1], heads, -1).transpose(1, 2)
        return (q, q, torch.ones(1)) if for_backward else q

    monkeypatch.setattr(ops, "q_proj", q_proj)
    monkeypatch.setattr(autograd, "_attn_forward", lambda q, k, v, *a, **kw: (q, k, v, torch.zeros_like(q), torch.zeros(8, 5)))
    monkeypatch.setattr(autograd, "_attn_backward", lambda do, q, k, v, *a, **kw: (torch.ones_like(q), torch.ones_like(k), torch.ones_like(v)))
    project_q = autograd.create_q_projection_class().apply
    w_q, w_kv = torch.randn(16, 8 * 4), torch.randn(16, 8 * 4, requires_grad=True)

    def run_function(x, states):
        k = (x @ w_kv).view(1, 5, 8, 4).transpose(1, 2)
        return project_q(x.detach(), w_q, 8, None, 1e-5), k, k

    x = torch.randn(1, 5, 16, requires_grad=True)
    autograd.create_attention_class("lv_xattn").apply(x, run_function, False).sum().backward()
    assert x.grad is not None and w_kv.grad is not None and calls == [False, False]


def test_a_checkpointed_projection_inside_run_function(monkeypatch):
    """A projection that run_function puts under torch.utils.checkpoint saves as many tensors in the attention's
    backward, where its gradient follows, as in the recomputation that checkpoint makes of it later: checkpoint
    refuses anything else."""
    from torch.utils.checkpoint import checkpoint
    raw = []

    def q_proj(x, w, heads, w_in_major=True, norm=None, eps=1e-5, for_backward=False):
        q = (x @ w).view(x.shape[0], x.shape[1], heads, -1).transpose(1, 2)
        raw.append(for_backward)
        return (q, q.clone(), torch.ones(1)) if for_backward else q

    def kv_proj(x, w_k, w_v, heads, w_in_major=True, k_norm_weight=None, eps=1e-5, for_backward=False):
        k, v = (q_proj(x, w, heads) for w in (w_k, w_v))
        return (k, v, k.clone(), torch.ones(1)) if for_backward else (k, v)

    monkeypatch.setattr(ops, "q_proj", q_proj)
    monkeypatch.setattr(ops, "kv_proj", kv_proj)
    monkeypatch.setattr(ops, "k_norm_bwd", lambda d, raw, r, w, want_dw: (d, torch.ones_like(w)))
    monkeypatch.setattr(ops, "q_proj_bwd", lambda x, d, w, *a, **kw: (torch.ones_like(x), torch.ones_like(w)))
    monkeypatch.setattr(ops, "dx_vis", lambda dk, dv, w_k, *a: torch.ones(1, 5, 16))
    monkeypatch.setattr(ops, "dw_kv", lambda x, dk, dv, *a: (torch.ones(16, 32), torch.ones(16, 32)))
    monkeypatch.setattr(autograd, "_attn_forward", lambda q, k, v, *a, **kw: (q, k, v, torch.zeros_like(q), torch.zeros(8, 5)))
    monkeypatch.setattr(autograd, "_attn_backward", lambda do, q, k, v, *a, **kw: (torch.ones_like(q), torch.ones_like(k), torch.ones_like(v)))
    project_q, project_kv = autograd.create_q_projection_class().apply, autograd.create_kv_projection_class().apply
    w_q, w_k, w_v = (torch.randn(16, 8 * 4, requires_grad=True) for _ in range(3))
    norm = torch.ones(4, requires_grad=True)

    def run_function(x, states):
        q = checkpoint(project_q, x, w_q, 8, norm, 1e-5, use_reentrant=False)
        return q, *checkpoint(project_kv, x, w_k, w_v, 8, norm, 1e-5, use_reentrant=False)

    x = torch.randn(1, 5, 16, requires_grad=True)
    autograd.create_attention_class("lv_xattn").apply(x, run_function, False).sum().backward()
    assert all(t.grad is not None for t in (x, w_q, w_k, w_v, norm)) and True in raw
