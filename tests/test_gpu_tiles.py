"""Tiles of tensors whose last but one dimension is contiguous, on either side of the sizes at which a CU holds two or three of them, at
1 bit (a wave per super-group) and the other widths, with ends inside a group, a super-group and a tile: against the same tensor made
contiguous first, bit for bit."""
import pytest
import torch

from gact import ops

pytestmark = pytest.mark.gpu


# batch, channels, pixels.  Tiles of 48 KB and 21 channels with one pixel fewer, or more, than they hold (half 1170, float 585), of 28 KB and
# small ones with tensors on either side of what takes them, one round and several, less than a tile
SHAPES = [(1, 8, 49), (3, 72, 50), (11, 128, 196), (47, 512, 784), (25, 640, 1169), (25, 640, 1171), (25, 640, 585), (25, 640, 586),
          (155, 512, 49), (188, 512, 49), (430, 512, 49), (130, 512, 405)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "%dx%dx%d" % s)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["f32", "f16", "bf16"])
def test_tiles_equal_the_contiguous_tensor(shape, dtype):
    b, c, k = shape
    x = torch.randn((b, k, c), generator=torch.Generator(device="cuda").manual_seed(k), device="cuda").to(dtype)
    x[0, : min(k, 300)] = 0.0
    x[0, k // 2, 3] = float("nan")
    x[-1, -1, -1] = 6e-8
    x = x.transpose(1, 2)
    y = x.contiguous()
    for bits in (1, 2, 4, 8):
        for stream in ("fast", "deterministic"):
            p, q = ops.op_quantize(x, bits, 5, rng_stream=stream), ops.op_quantize(y, bits, 5, rng_stream=stream)
            assert torch.equal(p[0][:-1], q[0][:-1]), (bits, stream)
            for got, ref in ((p[2], q[2]), (p[3], q[3])):
                assert torch.equal(got.nan_to_num(7.0), ref.nan_to_num(7.0)), (bits, stream)
