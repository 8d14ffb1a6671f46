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
