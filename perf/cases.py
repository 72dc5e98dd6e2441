"""The work a user has this framework do, as cases that can be timed and compared.

Every case goes through the public entry points of `lv_xattn`: `_attn_forward`, the autograd
wrappers of `lv_xattn.autograd` and the Hugging Face attention function.  The sizes are those of
the Llama-3.2-Vision cross-attention layers the repository is benchmarked on (32 query heads, 8
key/value heads of 128, images of four tiles of 1601 tokens, hidden size 4096), of the reference's
harness (16 heads, 1024 x 4096, fp16) and of its smaller head dimensions.

Run from the repository's root: the package under `lv-xattn_amd/` of the working folder is used.
"""
import math
import os
import sys
from types import SimpleNamespace

import torch

sys.path.insert(1, os.path.join(os.getcwd(), "lv-xattn_amd"))

import lv_xattn  # noqa: E402
from lv_xattn import autograd as lvx_autograd  # noqa: E402
from lv_xattn import hf_mllama  # noqa: E402

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
EPS = 1e-5                     # of the q and k norms


def _case(name, kind, **sizes):
    return dict(dict(kind=kind, B=1, Hq=32, Hkv=8, D=128, dtype="bf16"), **sizes, name=name)


def listed():
    return [
        # one new text token against the cached keys and values of one image, no mask: the latency
        # a generated token pays in every cross-attention layer
        _case("decode_token", "forward", Lq=1, Lkv=6404, rounds=1, merge=False),
        # generation through transformers: a batch of four, one token each, eight cross-attention
        # layers that share the mask transformers built for this token
        _case("hf_decode", "hf", B=4, Lq=1, Lkv=6404, layers=8),
        # the prompt of a batch of two through the same eight layers, with images of different length
        _case("hf_prefill", "hf", B=2, Lq=300, Lkv=6404, layers=8),
        # a short question (63 text tokens, the reference harness' length) about twelve images or a
        # video of that length: few rows, very many keys
        _case("prompt_long_video", "forward", Lq=63, Lkv=76848, rounds=1, merge=False),
        # the forward round loop of one GPU of sixteen: every visiting query block of 256 rows is
        # computed against the local shard and folded into the accumulator it brings along
        _case("prefill_rounds", "forward", Lq=4096, Lkv=6404, rounds=16, merge=True),
        # one training step of a whole cross-attention layer as the reference's harness calls it
        # (x, run_function): q, k, v projections with their norms, attention, and every gradient, the
        # projections recomputed in backward; a batch of two texts of ordinary, odd length
        _case("train_layer", "layer", B=2, Lq=1023, Lkv=6404, Dm=4096),
        # the flagship step: attention with key/value recompute from the visual states, dQ and dX_vis,
        # all query blocks in one launch
        _case("train_recompute", "recompute", Lq=4096, Lkv=6404, Dm=4096, rounds=16, batched=True),
        # the same work as the ring does it: one launch per visiting block, sixteen of them
        _case("train_rounds", "recompute", Lq=4096, Lkv=6404, Dm=4096, rounds=16, batched=False),
        # fine-tuning on a ragged batch: each text token sees the tiles of the image before it, the
        # second sample has less text and fewer tokens
        _case("train_masked", "attention", B=2, Lq=3000, Lkv=6404, image_tokens=3202, bias=False),
        # the reference's own harness: fp16, no head grouping, a dense additive bias
        _case("train_bias", "attention", Hq=16, Hkv=16, Lq=1024, Lkv=4096, dtype="fp16", image_tokens=0, bias=True),
        # a model with heads of 64
        _case("train_d64", "attention", D=64, Lq=2048, Lkv=6404, image_tokens=0, bias=False),
        # training on a long video's shard of 65536 visual tokens
        _case("train_long_video", "recompute", Lq=2048, Lkv=65536, Dm=4096, rounds=16, batched=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above: head groupings, head dimensions, both element types, text
    lengths from one row to 4096, shards from a tile or less to a long video, with and without masks."""
    limit = _cost(listed()[-1])
    while True:
        kind = rng.choice(["forward", "forward", "hf", "attention", "attention", "layer", "recompute"])
        hkv = rng.choice([1, 2, 4, 8, 8, 16])
        c = dict(kind=kind, B=rng.choice([1, 1, 2, 3, 4]), Hq=hkv * rng.choice([1, 2, 4, 4, 8]), Hkv=hkv,
                 D=rng.choice([128, 128, 128, 64, 64, 32, 16]), dtype=rng.choice(["bf16", "bf16", "fp16"]),
                 Lq=_log_int(rng, 1, 4096), Lkv=_log_int(rng, 400, 77000))
        if kind == "forward":
            c.update(rounds=rng.choice([1, 1, 4, 16]), merge=rng.random() < 0.5)
        elif kind == "hf":
            c.update(layers=rng.choice([1, 4, 8]), Lq=_log_int(rng, 1, 1024), Lkv=_log_int(rng, 400, 13000))
        elif kind == "attention":
            c.update(image_tokens=rng.choice([0, max(100, c["Lkv"] // rng.choice([1, 2, 3, 5]))]), bias=False)
            if rng.random() < 0.3:
                c.update(image_tokens=0, bias=True, Lkv=_log_int(rng, 400, 13000))
        elif kind == "layer":
            c.update(Dm=rng.choice([1024, 2048, 4096]), D=128)
        else:
            c.update(Dm=rng.choice([512, 1024, 2048, 4096]), rounds=rng.choice([1, 4, 16]), batched=rng.random() < 0.6)
        # small heads cost more per operation, so that they are counted as heads of 64
        if c["Hq"] <= 64 and _cost(dict(c, D=max(64, c["D"]))) <= limit / 2 and _bytes_held(c) < 8e9:
            return c


# ---------------------------------------------------------------------------------- masks
def _image_rows(case):
    """(first row, last row, first key, last key) per sample and image: the text rows that follow an
    image see its tokens and nothing else.  Later samples have less text and fewer images."""
    spans = []
    for b in range(case["B"]):
        n_text = max(1, case["Lq"] - b * (case["Lq"] * 2 // 5)) if b < 2 else max(1, case["Lq"] // 2)
        n_img = max(1, case["Lkv"] // case["image_tokens"] - b)
        first = n_text // 20                        # some text before the first image
        for i in range(n_img):
            lo = first + (n_text - first) * i // n_img
            hi = first + (n_text - first) * (i + 1) // n_img
            spans.append((b, lo, hi, i * case["image_tokens"], (i + 1) * case["image_tokens"]))
    return spans


def _visible_keys(case):
    """Keys each sample of the Hugging Face cases sees: whole tiles of 1601, or a share of the keys."""
    step = 1601 if case["Lkv"] >= 2 * 1601 else max(1, case["Lkv"] // 4)
    return [max(step, case["Lkv"] // step * step - (b % 3) * step) for b in range(case["B"])]


def _pairs(case):
    """Visible (text row, key) pairs per query head, over the batch."""
    if case["kind"] == "attention" and case["image_tokens"]:
        return sum((r1 - r0) * (k1 - k0) for _, r0, r1, k0, k1 in _image_rows(case))
    if case["kind"] == "hf":
        return case["Lq"] * sum(_visible_keys(case))
    return case["B"] * case["Lq"] * case["Lkv"]


# ---------------------------------------------------------------------------------- work
def work(case):
    """Bytes and operations of one pass: 4 D per visible pair and query head forward, 10 D backward, 2 M N K
    per projection product; every input read once, every output written once."""
    B, Hq, Hkv, D, Lq, Lkv = (case[k] for k in ("B", "Hq", "Hkv", "D", "Lq", "Lkv"))
    q, kv, lse = 2 * B * Hq * Lq * D, 2 * B * Hkv * Lkv * D, 4 * B * Hq * Lq
    pair = _pairs(case) * Hq * D
    if case["kind"] == "forward":
        return {"bytes": (2 * q + lse) * (2 if case["merge"] else 1) - (q if case["merge"] else 0) + 2 * kv, "flops": 4 * pair}
    if case["kind"] == "hf":
        seen = 2 * Hkv * D * sum(_visible_keys(case))
        return {"bytes": case["layers"] * (2 * q + 2 * seen) + 2 * B * Lq * Lkv, "flops": case["layers"] * 4 * pair}
    if case["kind"] == "attention":
        bias = 2 * 4 * Lq * Lkv if case["bias"] else 0
        return {"bytes": 4 * q + 4 * kv + bias, "flops": 14 * pair}
    Dm, N = case["Dm"], Hkv * D
    x_vis, w_kv = 2 * B * Lkv * Dm, 2 * 2 * Dm * N
    proj = 2 * 2 * B * Lkv * Dm * N                 # K and V: forward, again in backward, and dX_vis
    if case["kind"] == "recompute":
        return {"bytes": 4 * q + 2 * x_vis + w_kv, "flops": 14 * pair + 3 * proj}
    x, w_q = 2 * B * Lq * Dm, 2 * Dm * Hq * D
    proj_q = 2 * B * Lq * Dm * Hq * D
    return {"bytes": 2 * q + 2 * x + 2 * x_vis + 2 * (w_kv + w_q), "flops": 14 * pair + 4 * proj + 4 * proj_q}


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 5e12, w["flops"] / 1e15)


def _bytes_held(case):
    """Bytes of a case's tensors; a cache holds the keys that a mask hides as well."""
    held = work(case)["bytes"]
    if case["kind"] == "hf":
        held += 2 * case["B"] * case["Hkv"] * case["Lkv"] * case["D"] * 2 * case["layers"]
    return held


# ---------------------------------------------------------------------------------- inputs
def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    B, Hq, Hkv, D, Lq, Lkv = (case[k] for k in ("B", "Hq", "Hkv", "D", "Lq", "Lkv"))

    def normal(*shape, std=1.0):
        return torch.empty(*shape, dtype=dt, device=DEV).normal_(0.0, std, generator=g)

    s = SimpleNamespace(case=case, kind=case["kind"], scale=D ** -0.5)
    if s.kind == "forward":
        s.q, s.k, s.v = normal(B, Hq, Lq, D), normal(B, Hkv, Lkv, D), normal(B, Hkv, Lkv, D)
        s.acc = None
        if case["merge"]:           # what the block has gathered on its way here
            s.acc = (normal(B, Hq, Lq, D, std=0.05), torch.empty(B * Hq, Lq, device=DEV).normal_(9.0, 0.5, generator=g))
    elif s.kind == "hf":
        # the layer's projections leave tokens outermost; the cache keeps keys and values per head
        s.q = [normal(B, Lq, Hq, D).transpose(1, 2) for _ in range(case["layers"])]
        s.kv = [(normal(B, Hkv, Lkv, D), normal(B, Hkv, Lkv, D)) for _ in range(case["layers"])]
        s.mask = torch.zeros(B, 1, Lq, Lkv, dtype=dt, device=DEV)
        for b, n in enumerate(_visible_keys(case)):
            s.mask[b, :, :, n:] = torch.finfo(dt).min
        s.module = SimpleNamespace(k_norm=True, is_causal=False)
    elif s.kind == "attention":
        std = 0.5 if case["bias"] else 1.0
        s.q, s.k, s.v = (normal(*shape, std=std).requires_grad_() for shape in
                         ((B, Hq, Lq, D), (B, Hkv, Lkv, D), (B, Hkv, Lkv, D)))
        s.do = normal(B, Hq, Lq, D)
        s.bias, s.mask = None, None
        if case["bias"]:            # a position-dependent additive bias, shared by batch and heads
            s.bias = torch.empty(1, 1, Lq, Lkv, device=DEV).normal_(0.0, 1.0, generator=g)
        elif case["image_tokens"]:
            start = torch.zeros(B, Lq, dtype=torch.int32, device=DEV)
            end = torch.zeros_like(start)
            for b, r0, r1, k0, k1 in _image_rows(case):
                start[b, r0:r1], end[b, r0:r1] = k0, k1
            s.mask = lv_xattn.Mask(None, start, end)
        s.apply = lvx_autograd.create_attention_class_save_qkv("lv_xattn", rounds=1, batched=True).apply
    elif s.kind == "recompute":
        s.x_vis = normal(B, Lkv, case["Dm"]).requires_grad_()
        s.w_k, s.w_v = (normal(case["Dm"], Hkv * D, std=case["Dm"] ** -0.5) for _ in range(2))
        s.q, s.do = normal(B, Hq, Lq, D).requires_grad_(), normal(B, Hq, Lq, D)
        s.apply = lvx_autograd.create_attention_class("lv_xattn", rounds=case["rounds"], batched=case["batched"]).apply
    else:
        Dm = case["Dm"]
        s.x, s.x_vis = normal(B, Lq, Dm).requires_grad_(), normal(B, Lkv, Dm).requires_grad_()
        s.w_q = normal(Hq * D, Dm, std=Dm ** -0.5).requires_grad_()
        s.w_k, s.w_v = (normal(Hkv * D, Dm, std=Dm ** -0.5).requires_grad_() for _ in range(2))
        s.q_norm, s.k_norm = ((1.0 + normal(D, std=0.1)).requires_grad_() for _ in range(2))
        s.do = normal(B, Hq, Lq, D)
        s.apply = lvx_autograd.create_attention_class("lv_xattn", rounds=1, batched=True).apply
        q_proj = lvx_autograd.create_q_projection_class(w_in_major=False).apply
        kv_proj = lvx_autograd.create_kv_projection_class(w_in_major=False).apply

        def project(x, states):
            q = q_proj(x, s.w_q, Hq, s.q_norm, EPS)
            k, v = kv_proj(states, s.w_k, s.w_v, Hkv, s.k_norm, EPS)
            return q, k, v
        s.project = project
    return s


# ---------------------------------------------------------------------------------- one pass
def run(s):
    if s.kind == "forward":
        with torch.no_grad():
            _, _, _, o, lse = lv_xattn._attn_forward(s.q, s.k, s.v, False, s.scale, "lv_xattn", rounds=s.case["rounds"],
                                                     batched=s.case["rounds"] == 1, acc_in=s.acc)
        return o, lse
    if s.kind == "hf":
        with torch.no_grad():
            return [hf_mllama.lv_xattn_attention_forward(s.module, q, k, v, s.mask, scaling=s.scale)[0]
                    for q, (k, v) in zip(s.q, s.kv)]
    if s.kind == "attention":
        args = (_as_given, [s.bias], []) if s.bias is not None else (None, [], [])
        o = s.apply(s.q, s.k, s.v, False, s.scale, *args, s.mask)
        return (o.detach(), *torch.autograd.grad(o, (s.q, s.k, s.v), s.do))
    if s.kind == "recompute":
        o = s.apply(s.q, s.x_vis, s.w_k, s.w_v, s.case["Hkv"], s.scale)
        return (o.detach(), *torch.autograd.grad(o, (s.q, s.x_vis), s.do))
    leaves = (s.x, s.x_vis, s.w_q, s.w_k, s.w_v, s.q_norm, s.k_norm)
    for t in leaves:
        t.grad = None
    lvx_autograd.set_global_cross_attention_states(s.x_vis)
    o = s.apply(s.x, s.project, False)
    o.backward(s.do)
    return (o.detach(), *(t.grad for t in leaves))


def _as_given(bias):
    return bias


# ---------------------------------------------------------------------------------- tolerance
def tolerance(case):
    """Four times what the path's outputs are off by from the same computation in 64 bits: 3e-3 in bf16 and
    7e-4 in fp16 (whose small gradients leave its normal range), 6.5e-3 and 9e-4 where the query and
    key projections and their norms round as well."""
    layer = case["kind"] == "layer"
    if case["dtype"] == "bf16":
        return {"rel": 2.5e-2 if layer else 1.2e-2}
    return {"rel": 3.5e-3 if layer else 3e-3}
