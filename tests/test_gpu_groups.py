"""config.group_size 64, 128 and 512 on the one-pass kernels, against the oracle's minimax -> pack -> unpack on the
zero-padded tensor: codes, scale and restored values bit for bit, minimum by value.  Sizes end inside a chunk, a group, a
super-group, a span of 512 elements, a row's and a wave's share of them; the values include groups that are constant, so narrow
that a half scale overflows, and with NaN in them."""
import numpy as np
import pytest
import torch

import oracle
from gact import ops
from gact.conf import config
from gact.cpp_extension import minimax, quantization

pytestmark = pytest.mark.gpu

BITS = [1, 2, 4, 8]
MODES = {"deterministic": oracle.NOISE_CONST, "fast": oracle.NOISE_FAST, "inject": oracle.NOISE_INJECT}


@pytest.fixture(autouse=True)
def _restore_config():
    saved = config.group_size
    yield
    config.group_size = saved


def check(x_cpu, group, bits, stream, seed):
    config.group_size = group
    n = x_cpu.numel()
    N = -(-n // group)
    flat = np.zeros(N * group, dtype=x_cpu.numpy().dtype)
    flat[:n] = x_cpu.numpy().ravel()
    mn, mx = oracle.minimax(flat.reshape(N, group))
    sc = oracle.scale(mn, mx, bits)
    noise = torch.rand(N * group, generator=torch.Generator().manual_seed(seed)) if stream == "inject" else None
    want = oracle.pack(flat.reshape(N, 1, group), mn, sc, bits, MODES[stream], seed, None if noise is None else noise.numpy())
    if noise is None:
        q = ops.op_quantize(x_cpu.cuda(), bits, seed, rng_stream=stream)
    else:
        q = ops.op_quantize(x_cpu.cuda(), bits, seed, noise=noise.cuda())
    it = np.uint16 if flat.dtype == np.float16 else np.uint32
    where = "n %d" % n
    np.testing.assert_array_equal(q[3].cpu().numpy().ravel(), mn, err_msg=where)
    np.testing.assert_array_equal(q[2].cpu().numpy().ravel().view(it), sc.view(it), err_msg=where)
    np.testing.assert_array_equal(q[0].cpu().numpy().view(np.uint8)[: want.size], want, err_msg=where)
    out = ops.op_dequantize(q, x_cpu.shape).cpu().numpy()
    ref = oracle.unpack(want, bits, sc, mn, N, 1, group).ravel()[:n].reshape(x_cpu.shape)
    ok = ~np.isnan(ref)
    np.testing.assert_array_equal(np.isnan(out), ~ok, err_msg=where)
    np.testing.assert_array_equal(out[ok].view(it), ref[ok].view(it), err_msg=where)


@pytest.mark.parametrize("group", [64, 128, 512])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16], ids=["f32", "f16"])
@pytest.mark.parametrize("bits", BITS)
def test_one_pass_groups_equal_the_oracle(group, dtype, bits):
    g = torch.Generator().manual_seed(group + bits)
    for n in (1, group - 1, group, group + 1, 511, 513, 8 * group - 3, 8 * group + 5, 4096, 4 * 4096 + group + 9, 70001):
        x = torch.randn(n, generator=g)
        if n > 4 * group:
            x[:group] = 0.25                                    # constant
            x[group:2 * group] = 1.0 + x[group:2 * group].clamp(-1, 1) * 1e-7   # half: constant or one step wide
            x[2 * group:3 * group] *= 2e-7                      # half: subnormal, the scale overflows
            x[3 * group + 1] = float("nan")
        for stream in MODES:
            check(x.to(dtype), group, bits, stream, 31 + n)


@pytest.mark.parametrize("group", [64, 128, 512])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16], ids=["f32", "f16"])
def test_one_pass_groups_past_the_lines_of_the_launch(group, dtype):
    """2^26 elements and a little more: past every size at which the dequantize launch takes more per lane or caps its
    occupancy."""
    x = torch.randn((1 << 26) + 77, generator=torch.Generator().manual_seed(group)).to(dtype)
    for bits in BITS:
        check(x, group, bits, "fast", 5)


def _special(numel, group, dtype, gen):
    """Groups with NaN, infinities and the type's largest values in them, at the first and last element and everywhere, between
    ordinary ones."""
    big = torch.finfo(dtype).max
    x = torch.randn(numel, generator=gen)
    for i, v in enumerate((float("nan"), float("inf"), -float("inf"), big, -big, 2e30, -2e30, -0.0, 1e-45)):
        for j, at in enumerate((slice(0, 1), slice(group - 1, group), slice(0, group), slice(0, group, 2), slice(group // 2, group // 2 + 8))):
            x[(9 * j + i) * group + at.start:(9 * j + i) * group + at.stop:at.step or 1] = v
    x[45 * group:45 * group + 2] = torch.tensor([float("inf"), -float("inf")])
    x[46 * group:46 * group + 2] = torch.tensor([big, -big])
    x[47 * group:48 * group] = float("nan")
    x[47 * group + 3] = 1.0
    return x.to(dtype).cuda()


def _bits(t):
    return t.contiguous().view(-1).view(torch.uint8)


@pytest.mark.parametrize("group", [64, 128, 512])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16], ids=["f32", "f16"])
@pytest.mark.parametrize("bits", BITS)
def test_special_values_equal_the_extension_calls(group, dtype, bits):
    """Bit for bit what minimax, pack and unpack, which serve every group size, make of the zero-padded tensor."""
    config.group_size = group
    x = _special(50 * group + 7, group, dtype, torch.Generator().manual_seed(bits))
    groups = torch.cat([x, x.new_zeros(group - 7)]).view(51, group)
    mn, mx = minimax.minimax(groups)
    for stream in ("fast", "deterministic"):
        q = ops.op_quantize(x, bits, 3, rng_stream=stream)
        codes, scale = quantization.pack_single_precision(groups.view(51, 1, group), mn.view(51, 1, 1), mx.view(51, 1, 1), bits, True, 3,
                                                          rng_stream=stream)
        assert torch.equal(q[0][:-1], codes[:-1]), stream
        assert torch.equal(_bits(q[2]), _bits(scale)) and torch.equal(_bits(q[3]), _bits(mn)), stream
        want = quantization.unpack_single_precision(codes, bits, scale, mn.view(51, 1, 1), 51, 1, group).view(-1)[:x.numel()]
        out = ops.op_dequantize(q, x.shape)
        assert torch.equal(_bits(out), _bits(want)) or torch.equal(torch.isnan(out), torch.isnan(want)) \
            and torch.equal(out[~out.isnan()], want[~want.isnan()]), stream


@pytest.mark.parametrize("groups", [(1 << 14) - 1, 1 << 14, (1 << 14) + 1])
def test_long_deterministic_half_tensors_at_one_bit_in_groups_of_512(groups):
    """On either side of the size from which their codes are joined byte by byte, the last group short."""
    g = torch.Generator().manual_seed(groups)
    x = torch.randn(groups * 512 - 3, generator=g)
    x[:512] = 0.25                                     # constant
    x[512:1024] *= 2e-7                                # subnormal, the scale overflows
    x[1024], x[2048], x[3000] = float("nan"), float("inf"), -65504.0
    check(x.half(), 512, 1, "deterministic", 3)
