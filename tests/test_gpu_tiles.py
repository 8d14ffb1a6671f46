"""Tiles of tensors whose last but one dimension is contiguous, on either side of the sizes at which a tile holds 48 KB, 64 KB and more, at
1 bit (a wave per super-group) and the other widths, with ends inside a group, a super-group and a tile: against the same tensor made
contiguous first, bit for bit."""
import pytest
import torch

from gact import ops
from gact.cpp_extension import _abi

pytestmark = pytest.mark.gpu


# batch, channels, pixels: 28 channels a tile of 48 KB (half 24576 elements, float 12288) and 768 tiles, one more pixel or one fewer
# element, odd numbers of pixels, tensors of less than a tile
@pytest.mark.parametrize("shape", [(1, 8, 49), (3, 72, 50), (90, 256, 49), (11, 128, 196), (75, 256, 196), (33, 512, 784), (45, 256, 877),
                                   (45, 256, 878), (70, 256, 438), (70, 256, 439), (37, 512, 1024), (9, 264, 2025)],
                         ids=lambda s: "%dx%dx%d" % s)
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
