"""Tensors that are not contiguous, quantized where they lie, against the same tensor made contiguous first (whose kernels
the oracle pins): codes, scale and minimum bit for bit.  Layouts the kernels take (contiguous runs; the last but one dimension
contiguous) at sizes that end inside a group, a super-group and a tile, and layouts they decline."""
import ctypes

import pytest
import torch

from gact import ops
from gact.cpp_extension import _abi, quantization

pytestmark = pytest.mark.gpu


def _rc(x, bits, stream="fast"):
    """What the entry point answers for the layout, and its outputs."""
    n = -(-x.numel() // 256)
    codes = torch.empty(quantization.packed_numel(bits, n, 1, 256), dtype=torch.int8, device="cuda")
    scale = torch.empty(n, dtype=torch.float32 if x.dtype == torch.bfloat16 else x.dtype, device="cuda")
    mn = torch.empty(n, dtype=x.dtype, device="cuda")
    dims = ctypes.c_int64 * x.dim()
    rc = _abi.lib().gact_quantize_strided(x.data_ptr(), _abi.dtype_code(x.dtype), x.dim(), dims(*x.shape), dims(*x.stride()), bits,
                                          _abi.NOISE_MODES[stream], 5, None, codes.data_ptr(), scale.data_ptr(), mn.data_ptr(), None,
                                          torch.cuda.current_stream().cuda_stream)
    return rc, codes, scale, mn


def channels_last(n, c, h, w):
    return lambda g: torch.randn((n, c, h, w), generator=g).contiguous(memory_format=torch.channels_last)


def heads(b, s, h, d):
    return lambda g: torch.randn((b, s, h, d), generator=g).permute(0, 2, 1, 3)


def keys(b, s, h, d):
    return lambda g: torch.randn((b, s, h, d), generator=g).permute(0, 2, 3, 1)


# name -> (tensor on the CPU, whether the kernels take it at 16-byte pieces of 8 elements)
LAYOUTS = {
    "channels_last_7x7": (channels_last(3, 512, 7, 7), True),
    "channels_last_14x14": (channels_last(2, 256, 14, 14), True),
    "channels_last_28x28": (channels_last(1, 72, 28, 28), True),
    "channels_last_56x56": (channels_last(2, 64, 56, 56), True),
    "channels_last_45x45": (channels_last(5, 24, 45, 45), True),       # an odd number of pixels
    "channels_last_224x224": (channels_last(1, 8, 224, 224), True),     # a channel of more than a tile
    "channels_last_one_group": (channels_last(1, 8, 3, 3), True),
    "channels_last_rgb": (channels_last(4, 3, 32, 32), False),
    "matrix_transposed": (lambda g: torch.randn((1000, 328), generator=g).t(), True),
    "matrix_transposed_tall": (lambda g: torch.randn((24, 5000), generator=g).t(), True),
    "matrix_columns": (lambda g: torch.randn((777, 4 * 136), generator=g)[:, 136:2 * 136], True),
    "matrix_odd_columns": (lambda g: torch.randn((777, 500), generator=g)[:, 3:100], False),
    "heads_64": (heads(4, 197, 12, 64), True),
    "heads_80": (heads(2, 100, 4, 80), True),
    "heads_8": (heads(1, 3, 2, 8), True),
    "heads_20": (heads(2, 33, 3, 20), False),                           # 20 halves are not whole pieces (20 floats are)
    "qkv_query": (lambda g: torch.randn((3, 65, 3, 4, 32), generator=g).permute(2, 0, 3, 1, 4)[0], True),
    "keys_transposed": (keys(3, 77, 4, 32), True),
    "keys_transposed_sliced": (lambda g: torch.randn((3, 77, 8, 32), generator=g)[:, :, 2:6].permute(0, 2, 3, 1), True),
    "expanded": (lambda g: torch.randn((5, 1, 256), generator=g).expand(5, 7, 256), True),
    "rows_of_every_other": (lambda g: torch.randn((64, 300), generator=g)[:, ::2], False),
}


@pytest.mark.parametrize("layout", sorted(LAYOUTS))
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["f32", "f16", "bf16"])
def test_strided_equals_contiguous(layout, dtype):
    make, taken = LAYOUTS[layout]
    x_cpu = make(torch.Generator().manual_seed(len(layout)))
    # convert in the layout's own storage, so that the tensor on the GPU has the same strides
    x = torch.empty(0)
    base = x_cpu._base if x_cpu._base is not None else x_cpu
    x = base.to(dtype).cuda().as_strided(x_cpu.shape, x_cpu.stride(), x_cpu.storage_offset()) \
        if base is not x_cpu else x_cpu.to(dtype).cuda()
    assert x.stride() == x_cpu.stride() and not x.is_contiguous()
    y = x.contiguous()
    N = -(-x.numel() // 256)
    for bits in (1, 2, 4, 8):
        for stream in ("fast", "deterministic", "reference"):
            a, b = ops.op_quantize(x, bits, 11, rng_stream=stream), ops.op_quantize(y, bits, 11, rng_stream=stream)
            where = "%s %d bit %s" % (layout, bits, stream)
            assert torch.equal(a[0][:-1], b[0][:-1]), where
            assert torch.equal(a[2], b[2]) and torch.equal(a[3], b[3]), where
            assert torch.equal(ops.op_dequantize(a, x.shape), ops.op_dequantize(b, x.shape)), where
        # and the launch was not declined (or was, and fell back to the copy)
        assert _rc(x, bits)[0] == (0 if taken or (layout == "heads_20" and dtype == torch.float32) else _abi.ESHAPE), layout
    assert a[2].numel() == N


@pytest.mark.parametrize("dense", [False, True], ids=["transposed", "dense"])
def test_lazily_negated_view(dense):
    """Memory holds the values before the negation: it is resolved first."""
    x = torch.randn((1000, 328), generator=torch.Generator().manual_seed(2)).cuda()
    x = x if dense else x.t()
    a, b = ops.op_quantize(torch._neg_view(x), 4, 3), ops.op_quantize((-x).contiguous(), 4, 3)
    assert torch.equal(a[0][:-1], b[0][:-1]) and torch.equal(a[2], b[2]) and torch.equal(a[3], b[3])


def test_strided_large_tensors():
    """Sizes at which a workgroup's tile is the largest, with every XCD's runs of tiles and a ragged last one."""
    g = torch.Generator(device="cuda").manual_seed(1)
    for shape in ((5, 256, 112, 112), (40, 1000, 28, 28), (31, 64, 56, 56), (300, 2048, 7, 7)):
        x = torch.randn(shape, generator=g, device="cuda").to(torch.float16).contiguous(memory_format=torch.channels_last)
        for y in (x, x.float()):
            a, b = ops.op_quantize(y, 4, 3), ops.op_quantize(y.contiguous(), 4, 3)
            assert _rc(y, 4)[0] == 0, shape
            assert torch.equal(a[0][:-1], b[0][:-1]) and torch.equal(a[2], b[2]) and torch.equal(a[3], b[3]), shape
    x = torch.randn((64, 197, 12, 64), generator=g, device="cuda").to(torch.bfloat16).permute(0, 2, 1, 3)
    a, b = ops.op_quantize(x, 2, 3), ops.op_quantize(x.contiguous(), 2, 3)
    assert _rc(x, 2)[0] == 0
    assert torch.equal(a[0][:-1], b[0][:-1]) and torch.equal(a[2], b[2]) and torch.equal(a[3], b[3])


# batch, channels, pixels: channels that do not fill a strip, first super-groups at every offset, a ragged last group; strips cut
# into segments and not, more of them than the GPU holds at once, and numbers for which a step takes one group (half: 270 and, in
# three segments, 180 of 32 channels; float: 264 and 180 of 16)
@pytest.mark.parametrize("shape", [(3, 40, 2052), (1, 8, 1540), (9, 40, 12292), (270, 32, 2048), (530, 32, 2060), (70, 256, 3076),
                                   (270, 32, 3076), (180, 32, 3076), (264, 16, 3076), (180, 16, 3076)], ids=lambda s: "%dx%dx%d" % s)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["f32", "f16", "bf16"])
def test_strips_of_long_channels(shape, dtype):
    b, c, k = shape
    x = torch.randn((b, k, c), generator=torch.Generator(device="cuda").manual_seed(k), device="cuda").to(dtype)
    x[0, :600] = 0.0        # groups of equal values: the largest scale there is (half: infinite in the first)
    x[0, 5, 0] = 6e-8
    x = x.transpose(1, 2)
    y = x.contiguous()
    for bits in (1, 2, 4, 8):
        for stream in ("fast", "deterministic"):
            p, q = ops.op_quantize(x, bits, 5, rng_stream=stream), ops.op_quantize(y, bits, 5, rng_stream=stream)
            assert _rc(x, bits, stream)[0] == 0
            assert torch.equal(p[0][:-1], q[0][:-1]) and torch.equal(p[2], q[2]) and torch.equal(p[3], q[3]), (bits, stream)


# [batch, channels, pixels], dtype, widths the kernels take in place, widths left to the contiguous copy, which is the faster way there
@pytest.mark.parametrize("shape,dtype,taken,declined", [
    ((4096, 8, 2), torch.float32, (1, 2, 4, 8), ()), ((1 << 19, 8, 2), torch.float32, (), (1, 2, 4, 8)),        # few pixels
    ((1 << 18, 64, 3), torch.float16, (2, 4, 8), (1,)), ((1 << 16, 64, 9), torch.float32, (2, 4, 8), (1,)),
    ((1 << 14, 64, 17), torch.float32, (1, 2, 4, 8), ()),
    ((1, 8, 20001), torch.float16, (1, 2, 4, 8), ()), ((3, 64, 20001), torch.float16, (), (1, 2, 4, 8)),        # long channels
    ((13, 64, 20001), torch.bfloat16, (1, 2, 4, 8), ()), ((7, 64, 20001), torch.float32, (1, 2, 4, 8), ()),
    ((1, 256, 50257), torch.float32, (), (1, 2, 4, 8)), ((42, 8, 12321), torch.float16, (), (1, 2, 4, 8)),
    ((83, 8, 12544), torch.float16, (2, 4, 8), (1,)), ((83, 8, 50176), torch.float16, (1, 2, 4, 8), ()),        # channels of one piece
    ((545, 8, 3844), torch.bfloat16, (1, 2, 4, 8), ()), ((700, 4, 3136), torch.float32, (1, 2, 4, 8), ()),
], ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v)[6:])
def test_where_the_contiguous_copy_is_faster_it_is_made(shape, dtype, taken, declined):
    b, c, k = shape
    x = torch.randn((b, k, c), generator=torch.Generator(device="cuda").manual_seed(k), device="cuda").to(dtype).transpose(1, 2)
    for bits in taken + declined:
        q = ops.op_quantize(x.contiguous(), bits, 5)
        rc, codes, scale, mn = _rc(x, bits)
        assert rc == (_abi.ESHAPE if bits in declined else 0), bits
        p = ops.op_quantize(x, bits, 5)
        for codes, scale, mn in [(p[0], p[2], p[3])] + ([(codes, scale, mn)] if bits in taken else []):
            assert torch.equal(codes[:-1], q[0][:-1]) and torch.equal(scale.view(-1), q[2].view(-1)) and torch.equal(mn.view(-1), q[3].view(-1)), bits


# one shape per kernel: pieces with addresses of their own, a tile, strips of one and of two groups per step (half, float)
@pytest.mark.parametrize("shape", [(40, 8, 784), (3, 40, 2052), (9, 40, 12292), (270, 32, 3076), (257, 16, 3076), (33, 12, 197, 64)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["f32", "f16", "bf16"])
def test_special_values(shape, dtype):
    """NaN, infinities and the largest values in single elements, in runs along the memory and along a channel, and in whole
    groups."""
    g = torch.Generator(device="cuda").manual_seed(sum(shape))
    x = torch.randn([shape[0], shape[2], shape[1]] + list(shape[3:]), generator=g, device="cuda").to(dtype).transpose(1, 2)
    big = torch.finfo(dtype).max
    for i, v in enumerate((float("nan"), float("inf"), -float("inf"), big, -big, 2e30 if dtype != torch.float16 else 6e-8, -0.0)):
        flat = torch.randint(0, x.numel(), (12,), generator=g, device="cuda")
        y = x.reshape(-1)               # a copy in index order
        y[flat] = v
        y[4096 * i + 1024:4096 * i + 1024 + 512] = v
        y[4096 * i + 2048:4096 * i + 2048 + 512:2] = v
        x.copy_(y.view(x.shape))
        x[0, i % shape[1], :40] = v
    y = x.contiguous()
    for bits in (1, 2, 4, 8):
        for stream in ("fast", "deterministic"):
            p, q = ops.op_quantize(x, bits, 5, rng_stream=stream), ops.op_quantize(y, bits, 5, rng_stream=stream)
            for a, b in ((p[0][:-1], q[0][:-1]), (p[2], q[2]), (p[3], q[3])):
                assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8)), (bits, stream)
