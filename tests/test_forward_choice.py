"""The ranges a forward launch is cut into: where the closer fit takes over from the first (us, first -> closer), and where it does not."""
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
