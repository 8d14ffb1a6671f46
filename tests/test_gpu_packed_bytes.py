"""Codes at the ends of the conversion that packs them, against the oracle bit for bit (no tolerance: the codes are whole numbers):
half groups whose largest element lands one code above its field (the scale is rounded to half), scales that overflow to infinity,
infinite and NaN elements, and the top code of float groups, at every width and stream, contiguous, in other group sizes and strided."""
import numpy as np
import pytest
import torch

import oracle
from gact import ops
from gact.conf import config

pytestmark = pytest.mark.gpu

MODES = {"deterministic": oracle.NOISE_CONST, "reference": oracle.NOISE_REF, "fast": oracle.NOISE_FAST}


@pytest.fixture(autouse=True)
def _restore_config():
    saved = config.group_size
    yield
    config.group_size = saved


def edge_values(n, dtype, bits, group):
    """n elements, half of every group at its maximum; from group to group a range whose largest half product lies above the
    largest code, a scale of infinity, an infinite element, a NaN, plain values."""
    g = np.random.default_rng(bits)
    x = g.random(n).astype(np.float32)
    q = np.float32(2 ** bits - 1)
    ranges = np.arange(64, 4000, dtype=np.float32) / 512
    half = ranges.astype(np.float16)
    scale = (np.float64(q) / (half.astype(np.float64) + 2e-6)).astype(np.float32).astype(np.float16)
    above = half[(half * scale).astype(np.float32) > q]
    assert bits == 1 or above.size > 20     # at 1 bit the product rounds back to 1
    above = above if above.size else half
    for k, first in enumerate(range(0, n, group)):
        part = x[first:first + group]
        r = np.float32(above[k % above.size])
        part *= r
        part[::2] = r
        part[1] = 0
        if k % 5 == 1:
            part *= np.float32(1e-6) / r       # half: subnormal, the scale overflows
        elif k % 5 == 2 and k % 10 == 2:
            part[g.integers(part.size)] = np.inf
        elif k % 5 == 3:
            part[g.integers(part.size)] = np.nan
    with np.errstate(over="ignore"):
        return torch.from_numpy(x).to(dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("bits", [1, 2, 4, 8])
@pytest.mark.parametrize("stream", list(MODES))
@pytest.mark.parametrize("n", [256 * 67, 256 * 4099 + 31])   # row and wave per super-group, staged and ragged rows
def test_edge_codes_equal_the_oracle(dtype, bits, stream, n):
    x = edge_values(n, dtype, bits, 256)
    want = oracle.op_quantize(x.float().numpy() if dtype == torch.bfloat16 else x.numpy(), bits, MODES[stream], 7)
    q = ops.op_quantize(x.cuda(), bits, 7, rng_stream=stream)
    np.testing.assert_array_equal(q[0].cpu().numpy().view(np.uint8)[: want[0].size], want[0])


@pytest.mark.parametrize("group", [64, 128, 512])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16], ids=["f32", "f16"])
@pytest.mark.parametrize("bits", [1, 2, 4, 8])
@pytest.mark.parametrize("stream", ["deterministic", "fast"])
def test_edge_codes_of_other_groups_equal_the_oracle(group, dtype, bits, stream):
    n = group * 133
    x = edge_values(n, dtype, bits, group)
    mn, mx = oracle.minimax(x.numpy().reshape(-1, group))
    want = oracle.pack(x.numpy().reshape(-1, 1, group), mn, oracle.scale(mn, mx, bits), bits, MODES[stream], 7)
    config.group_size = group
    q = ops.op_quantize(x.cuda(), bits, 7, rng_stream=stream)
    np.testing.assert_array_equal(q[0].cpu().numpy().view(np.uint8)[: want.size], want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("bits", [1, 2, 4, 8])
@pytest.mark.parametrize("shape", [(2, 64, 64, 64), (2, 64, 16, 16)], ids=["strips", "tiles"])
def test_edge_codes_of_strided_tensors_equal_the_oracle(dtype, bits, shape):
    x = edge_values(int(np.prod(shape)), dtype, bits, 256).view(shape)
    want = oracle.op_quantize(x.float().numpy() if dtype == torch.bfloat16 else x.numpy(), bits, oracle.NOISE_FAST, 7)
    q = ops.op_quantize(x.cuda().contiguous(memory_format=torch.channels_last), bits, 7, rng_stream="fast")
    np.testing.assert_array_equal(q[0].cpu().numpy().view(np.uint8)[: want[0].size], want[0])
