"""The rules for tensors that are quantized where they lie (strided_rules.py), and that the shapes of the GPU tests take every branch of them."""
import itertools

import pytest

import strided_rules
import test_gpu_strip_stats
import test_gpu_tiles

SIZES = (2, 4)
BITS = (1, 2, 4, 8)


def up(n, d):
    return -(-n // d)


def cut(slots, most, numel):
    return up(up(numel, slots * up(numel, slots * most)), 2048) * 2048


def ways(size, bits, numel, k):
    """Tiles for two workgroups of a CU (or one) and for three, and whether those for three are the ones to take."""
    two = cut(256, 147456 // size, numel) if min(65536 // size, numel // 512) < 16 * k else cut(512, 65536 // size, numel)
    three = cut(768, 49152 // size, numel)
    two_on, three_on = (up(up(numel, t), 256) * t for t in (two, three))     # elements on the CU that gets most
    return two, three, not (size == 4 and bits == 2) and three >= 21 * k and (three * size >= 28 * 1024 or three_on <= two_on)


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("bits", BITS)
def test_what_a_tile_is_left_with_decides(size, bits):
    """A third workgroup on a CU pays for tiles that still hold many channels when the tensor has been cut: half [87,256,876] at 2 bit,
    28 KB and 16 channels a tile, took 19.6 us where tiles of 40 KB take 17.6."""
    for k, millions in itertools.product((9, 49, 100, 196, 400, 585, 600, 784, 876, 1170, 1225), range(1, 120)):
        numel = millions * 500000 // (8 * k) * 8 * k
        two, three, by_threes = ways(size, bits, numel, k)
        assert strided_rules.rules().tile(size, bits, numel, k) == (three if by_threes else two), (k, numel)


def test_the_shapes_of_the_tile_test_take_both_kinds_of_tiles():
    for size, bits in itertools.product(SIZES, BITS):
        seen = set()
        for shape in test_gpu_tiles.SHAPES:
            b, c, k = shape
            tile = strided_rules.tile(size, bits, shape)
            assert tile or k % 4 == 0                                   # strips take multiples of four pixels only
            if tile and b * c * k >= 1 << 20:
                three = ways(size, bits, b * c * k, k)[2]
                seen.add((three, "48 KB" if tile * size == 49152 else "36 KB" if tile * size >= 36864 else "less", b * c * k > (768 if three else 512) * tile))
        assert any(not three and size_ != "less" for three, size_, _ in seen)
        if not (size == 4 and bits == 2):
            assert (True, "48 KB", False) in seen and any(three and many for three, _, many in seen), seen


def test_the_shapes_of_the_strip_test_are_strips():
    seen = set()
    for shape, size, bits in test_gpu_strip_stats.CASES:
        cut = strided_rules.strip_cut(size, bits, shape)
        assert cut, (shape, size, bits)
        seen.add((size, bits, cut[0]))
        if cut[1] > 1:
            seen.add((size, bits, "segments"))
    for size, bits in itertools.product(SIZES, BITS):
        assert {(size, bits, 1), (size, bits, "segments")} <= seen and ((size, bits, 2) in seen or bits == 8), (size, bits)
