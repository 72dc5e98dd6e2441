"""The ranges a forward launch is cut into: where the closer fit takes over from the first (us, first -> closer), and where it does not."""
import math
import random

import pytest


@pytest.mark.parametrize("shape,ranges", [
    ((4, 8, 8, 36, 58268, 128), 4),                 # few rows of many keys, 215 -> 169
    ((1, 8, 2, 1, 670, 64), 11),                    # a short shard, 8.9 -> 6.4
    ((1, 32, 8, 1, 6404, 128), 29), ((4, 32, 8, 1, 6404, 128), 8),      # within 12 % of each other: as before
    ((2, 32, 8, 300, 6404, 128), 3), ((1, 32, 8, 256, 6404, 128), 8), ((1, 32, 8, 4096, 6404, 128), 1)])
def test_ranges_of_a_launch(shape, ranges):
    from lv_xattn.attn import auto_kv_splits
    assert auto_kv_splits(*shape) & 255 == ranges


def test_parts_that_were_not_there_before_wait_in_fp32():
    """Launches that the first fit leaves whole and the closer one cuts: an O in 16-bit parts would be a rounding more."""
    from lv_xattn.attn import auto_kv_splits
    for shape in [(4, 8, 2, 24, 749, 64), (4, 16, 4, 706, 9539, 128), (2, 64, 8, 303, 4410, 16), (1, 32, 16, 1129, 3353, 32)]:
        n = auto_kv_splits(*shape)
        assert n == 1 or n & 256


def _first_fit(B, Hq, Hkv, rows, Lkv, D, bias=False, cus=256):
    """The number of ranges that the first fit finds cheapest, and whether their parts wait in fp32.  With a dense bias: of the plain form, at
    the price it has without one."""
    G = Hq // Hkv
    hg = math.gcd(G, 4)
    wide = D in (64, 128) and not bias

    def cost(few, splits, f32):
        step = 32 if few else 64
        length = -(-(-(-Lkv // splits)) // step) * step
        n = -(-Lkv // length)
        us = 4.0 + n * B * Hq * rows * ((4 * D + 8) / 4e6 + (4 * D / 9e6 if f32 else 0.0)) if n > 1 else 0.0
        if few:
            wgs, slots = B * Hkv * -(-rows * G // 32) * n, cus if D == 128 else 2 * cus
            key_us = {128: 8e-3, 64: 4.2e-3}.get(D, 3e-3)
            return us + 5.0 + math.hypot(-(-wgs // slots) * (length * key_us + 3.0) - 3.0, B * Hkv * Lkv * D * 4 / 5.2e6)
        wgs, slots = B * (Hq // hg) * -(-rows // ((64 if wide else 32) * (4 // hg))) * n, cus if wide else 2 * cus
        tile_us, load_us = (0.8, 1.0) if not wide else (1.1, 0.4) if D == 128 else (0.9, 0.15)
        return us + -(-wgs // slots) * (length // 64 * (tile_us + load_us * min(1.0, wgs / slots)) + 11.0)

    few_f32, many_f32 = True, B * (Hq // hg) * -(-rows // (32 * (4 // hg))) >= 2 * cus or Lkv < 1024
    return min((cost(few, n, f32), few, n, n > 1 and f32) for few, f32 in ((False, many_f32), (True, few_f32)) if not few or (rows * G <= 256 and not bias)
               for n in range(1, 65) if n == 1 or Lkv // n >= 32)[2:]


def _launches(seed, count, most_keys):
    rng = random.Random(seed)

    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    for _ in range(count):
        hkv = rng.choice([1, 2, 4, 8, 8, 16])
        yield (rng.choice([1, 1, 2, 3, 4]), hkv * rng.choice([1, 2, 4, 4, 8]), hkv, log_int(1, 4096), log_int(300, most_keys),
               rng.choice([128, 128, 128, 64, 64, 32, 16]))


def _held_in_16_bits(n):
    return n > 1 and not n & 256


def test_no_part_waits_in_fewer_bits_than_the_first_fit_says():
    from lv_xattn.attn import auto_kv_splits
    few_to_wide = [(2, 32, 8, 45, 3450, 128), (1, 8, 8, 206, 7423, 128), (1, 32, 8, 49, 62466, 64), (4, 4, 4, 250, 20294, 64),
                   (3, 8, 2, 62, 25098, 64), (1, 16, 16, 188, 46687, 64), (3, 4, 4, 220, 5649, 128)]
    assert [_first_fit(*s) for s in few_to_wide[:2]] == [(2, True), (4, True)]
    for shape in few_to_wide + list(_launches(11, 6000, 77000)):
        n, f32 = _first_fit(*shape)
        assert not _held_in_16_bits(auto_kv_splits(*shape)) or (n > 1 and not f32), shape


def test_no_part_of_a_launch_with_a_bias_waits_in_fewer_bits_than_the_plain_form_says():
    from lv_xattn.attn import auto_kv_splits
    left_whole = [(1, 32, 4, 638, 1059, 128), (1, 8, 1, 1903, 1090, 128), (1, 64, 8, 293, 1095, 128), (1, 64, 8, 254, 1251, 128),
                  (3, 16, 8, 441, 1563, 128), (3, 64, 16, 96, 1024, 64)]
    for shape in left_whole + list(_launches(12, 6000, 13000)):
        n, f32 = _first_fit(*shape, bias=True)
        assert shape not in left_whole or n == 1
        assert not _held_in_16_bits(auto_kv_splits(*shape, True)) or (n > 1 and not f32), shape


@pytest.mark.parametrize("shape,most", [         # us with so many ranges, with those of a price without what a part costs
    ((3, 1, 1, 142, 3391, 128), 40),                # 27: 14.5, 53: 18.3
    ((1, 4, 1, 198, 3374, 64), 40),                 # 27: 12.9, 53: 15.6
    ((4, 8, 2, 40, 1151, 128), 14),                 # 9: 15.2, 18: 17.8
    ((4, 4, 1, 39, 7360, 128), 40), ((2, 8, 2, 75, 4281, 128), 26), ((1, 8, 2, 160, 4018, 64), 26), ((1, 8, 8, 739, 860, 64), 6)])
def test_a_launch_with_a_bias_is_not_cut_for_less_than_its_parts_cost(shape, most):
    from lv_xattn.attn import auto_kv_splits
    assert 1 < auto_kv_splits(*shape, True) & 255 <= most


@pytest.mark.parametrize("shape", [             # us with the first fit's ranges, with those of one price per key and part
    (3, 16, 16, 155, 2652, 64),                     # 17.5, 19.8
    (1, 8, 8, 167, 1018, 64),                       # 8.6, 9.5
    (4, 16, 4, 58, 1347, 64), (3, 8, 1, 5, 955, 64), (2, 16, 8, 35, 1141, 64),
    (2, 2, 2, 3, 12498, 32),                        # 7.5, 8.6
    (1, 8, 4, 1, 11309, 32), (1, 2, 2, 2, 10552, 32), (4, 1, 1, 2, 7849, 32)])
def test_short_launches_and_small_heads_keep_the_ranges_of_the_first_fit(shape):
    from lv_xattn.attn import auto_kv_splits
    n, f32 = _first_fit(*shape)
    assert auto_kv_splits(*shape) == n | 256 * f32
