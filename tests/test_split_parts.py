"""Key splits whose parts are fp32: the sizes and refusals of the C entry points, checked without a GPU."""
import ctypes as C

import pytest

F32 = 256


def _shape(**kw):
    from lv_xattn import _lib
    s = dict(B=1, Hq=32, Hkv=8, D=128, Lq=4096, Lkv=6404, dtype=_lib.LVX_BF16, scale=1.0)
    return _lib.AttnShape(*dict(s, **kw).values())


def test_fp32_parts_need_twice_the_room_for_o():
    from lv_xattn import _lib
    lib = _lib.load()
    s = _shape()
    for n in (2, 64):
        assert lib.lvx_fwd_workspace_bytes(C.byref(s), 100, n) == n * 32 * 100 * (128 * 2 + 4)
        assert lib.lvx_fwd_workspace_bytes(C.byref(s), 100, n | F32) == n * 32 * 100 * (128 * 4 + 4)
    for n in (1, 0, -1, 1 | F32, F32):
        assert lib.lvx_fwd_workspace_bytes(C.byref(s), 100, n) == 0


@pytest.mark.parametrize("entry", ["lvx_fwd", "lvx_fwd_noalloc"])
@pytest.mark.parametrize("splits,code", [(0, -3), (65, -3), (F32, -3), (65 | F32, -3), (512, -3), (-1, -3), (-F32, -3), (4, -7), (4 | F32, -7)])
def test_only_1_to_64_splits_are_taken_and_their_room_is_checked(entry, splits, code):
    from lv_xattn import _lib
    lib = _lib.load()
    s = _shape()
    t = _lib.Tensor4(0x1000, 32 * 4096 * 128, 4096 * 128, 128)
    args = [C.byref(s)] + [C.byref(t)] * 4 + [0x2000, 0, 4096, splits]
    if entry == "lvx_fwd":
        args += [0x3000, lib.lvx_fwd_workspace_bytes(C.byref(s), 4096, splits) - 1 if code == -7 else 1 << 40]
    assert getattr(lib, entry)(*args, None) == code


# (rows, keys, bias): what is chosen stays in 16 bits only where a launch of 32- or 64-row waves cannot fill the chip
@pytest.mark.parametrize("Lq,Lkv,kw,f32", [
    (1, 6404, {}, True), (25, 929, {}, True), (256, 929, {}, True), (256, 6404, {}, False), (63, 76848, {}, False),
    (2100, 6404, {}, True), (2100, 6404, dict(D=32), True), (256, 929, dict(D=32), True), (256, 6404, dict(D=32), False),
    (256, 6404, dict(bias=16), False), (2100, 6404, dict(bias=16), True)])
def test_splits_chosen_by_the_library(Lq, Lkv, kw, f32):
    from lv_xattn import _lib
    s = _shape(Lq=Lq, Lkv=Lkv, **{k: v for k, v in kw.items() if k != "bias"})
    if "bias" in kw:
        s.bias, s.bias_stride_r = 16, (Lkv + 3) // 4 * 4
    n = _lib.load().lvx_fwd_auto_splits(C.byref(s), Lq)
    assert 2 <= n & (F32 - 1) <= 64 and bool(n & F32) == f32
