"""Strips of channels-last tensors keep the scales and minima of several steps before they store them: channels that end inside such a
turn, strips cut into segments that begin inside one, a ragged end, against the same tensor made contiguous first: bit for bit, and
nothing written beside them."""
import pytest
import torch

from gact import ops
from gact.cpp_extension import _abi, quantization

import ctypes

pytestmark = pytest.mark.gpu


DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
# batch, channels, pixels; 1 and 2 bit take strips where tensors are large
SMALL = [(1, 16, 2048), (1, 24, 4100), (3, 40, 5636), (1, 64, 12544)]
LARGE = [(1, 64, 65540), (3, 40, 36868), (60, 72, 4096), (130, 32, 4356)]
CASES = [(shape, 4 if name == "f32" else 2, bits) for name in DTYPES for bits in (1, 2, 4, 8) for shape in (SMALL if bits >= 4 else []) + LARGE]
PARAMS = [pytest.param(shape, name, bits, id="%dx%dx%d-%s-%d" % (*shape, name, bits))
          for name in DTYPES for bits in (1, 2, 4, 8) for shape in (SMALL if bits >= 4 else []) + LARGE]


@pytest.mark.parametrize("shape, dtype, bits", PARAMS)
def test_scales_and_minima_of_strips(shape, dtype, bits):
    dtype = DTYPES[dtype]
    b, c, k = shape
    g = torch.Generator(device="cuda").manual_seed(k + bits)
    x = torch.randn((b, k, c), generator=g, device="cuda").to(dtype).permute(0, 2, 1)
    n = -(-x.numel() // 256)
    room = 64
    codes = torch.empty(quantization.packed_numel(bits, n, 1, 256), dtype=torch.int8, device="cuda")
    scale = torch.full((n + 2 * room,), 7.0, dtype=torch.float16 if dtype is torch.float16 else torch.float32, device="cuda")
    mn, mx = (torch.full((n + 2 * room,), 7.0, dtype=dtype, device="cuda") for _ in range(2))
    dims = ctypes.c_int64 * 3
    at = [t.data_ptr() + room * t.element_size() for t in (scale, mn, mx)]
    rc = _abi.lib().gact_quantize_strided(x.data_ptr(), _abi.dtype_code(dtype), 3, dims(*x.shape), dims(*x.stride()), bits, _abi.NOISE_FAST, 5,
                                          None, codes.data_ptr(), *at, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    want = ops.op_quantize(x.contiguous(), bits, 5, rng_stream="fast")
    for got, ref in ((scale, want[2]), (mn, want[3])):
        assert torch.equal(got[room:room + n], ref.flatten())
        assert bool((got[:room] == 7.0).all()) and bool((got[room + n:] == 7.0).all())
    flat = torch.zeros(n * 256, dtype=dtype, device="cuda")
    flat[:x.numel()] = x.reshape(-1)
    assert torch.equal(mx[room:room + n], flat.view(n, 256).max(dim=1).values)
    assert bool((mx[:room] == 7.0).all()) and bool((mx[room + n:] == 7.0).all())
    assert torch.equal(codes[:-1], want[0][:-1])
