"""The Hugging Face attention function's host side, with the kernels replaced by stand-ins: what it
refuses, what it hands to autograd."""
import pytest
import torch
from torch.autograd import forward_ad

from lv_xattn import autograd, hf_mllama


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
