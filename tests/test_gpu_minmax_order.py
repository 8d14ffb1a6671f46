"""Minima and maxima by the packed three-operand instructions of half (and of bfloat16 where its bits are ordered as half's are), which
hand a NaN on where the reference ignores it: groups with NaN, infinities, zeros of both signs, subnormals and, for bfloat16, values
beyond 2^121 (which look like a half NaN) and beyond the reference's start value 1e30, next to groups without, through
every kernel that takes them: whole and ragged tensors, strided ones, batches.  Against the oracle: all bit for bit, the
minimum by value."""
import numpy as np
import pytest
import torch

import oracle
from gact import ops
from gact.batched import BatchedQuantizer

pytestmark = pytest.mark.gpu

SPECIAL = {"nan": float("nan"), "inf": float("inf"), "-inf": float("-inf"), "-0": -0.0, "subnormal": 6e-8}
WIDE = {"2^120": 2.0 ** 120, "2^121": 2.0 ** 121, "-2^122": -(2.0 ** 122), "max": 3.3e38, "tiny": 1e-39}


def values(n, dtype, seed):
    """Every third group of 256 holds one special value in one place, every seventh is made of one throughout."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(n, generator=g)
    special = list((dict(SPECIAL, **WIDE) if dtype is torch.bfloat16 else SPECIAL).values())
    for k, at in enumerate(range(0, n, 3 * 256)):
        x[min(n - 1, at + int(torch.randint(0, 256, (1,), generator=g)))] = special[k % len(special)]
    for k, at in enumerate(range(512, n, 7 * 256)):
        x[at:at + 256] = special[k % len(special)]
    x[1024:1280] = torch.where(x[1024:1280] > 0, 0.0, -0.0)
    return x.to(dtype)


def want(x, bits, mode, seed):
    wide = x.float() if x.dtype is torch.bfloat16 else x
    with np.errstate(all="ignore"):
        return oracle.op_quantize(np.ascontiguousarray(wide.numpy()), bits, mode, seed)


def same(q, ref, tag):
    it = np.uint32 if ref[2].dtype == np.float32 else np.uint16
    mn, got = ref[3].ravel(), q[3].float().cpu().numpy().ravel()
    ok = ~np.isnan(mn.astype(np.float32))
    # bfloat16 keeps the minimum in 16 bits: the start value 1e30 of a group without a smaller element is the only one that rounds
    if q[3].dtype is torch.bfloat16:
        mn = torch.from_numpy(mn.astype(np.float32)).to(torch.bfloat16).float().numpy()
    np.testing.assert_array_equal(got[ok], mn[ok].astype(np.float32), err_msg=tag)
    np.testing.assert_array_equal(q[2].cpu().numpy().ravel().view(it), ref[2].ravel().view(it), err_msg=tag)
    np.testing.assert_array_equal(q[0].cpu().numpy().view(np.uint8)[: ref[0].size], ref[0], err_msg=tag)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("bits", [1, 2, 4, 8])
def test_contiguous_tensors(dtype, bits):
    for n in (2048, 8 * 256 * 9 + 77, 256 * 41000 + 3):    # the last: past the wave-per-super-group form at 1 bit
        x = values(n, dtype, bits)
        for mode, stream in ((oracle.NOISE_CONST, "deterministic"), (oracle.NOISE_FAST, "fast"), (oracle.NOISE_REF, "reference")):
            same(ops.op_quantize(x.cuda(), bits, 7, rng_stream=stream), want(x, bits, mode, 7), "%d %s" % (n, stream))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("bits", [1, 4])
@pytest.mark.parametrize("layout", ["heads", "tiles", "strips"])
def test_strided_tensors(dtype, bits, layout):
    shape = {"heads": (2, 4, 100, 64), "tiles": (2, 64, 14, 14), "strips": (2, 64, 64, 64)}[layout]
    x = values(int(np.prod(shape)), dtype, bits + 20).reshape(shape)
    strided = x.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3) if layout == "heads" else x.contiguous(memory_format=torch.channels_last)
    same(ops.op_quantize(strided.cuda(), bits, 7, rng_stream="fast"), want(x, bits, oracle.NOISE_FAST, 7), layout)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
def test_batches(dtype):
    sizes, widths = [256 * 131 + 5, 4096, 70001, 300], [1, 2, 4, 8]
    xs = [values(n, dtype, 40 + n % 7) for n in sizes]
    on_gpu = [x.cuda() for x in xs]
    batch = BatchedQuantizer(sizes, [dtype] * len(xs), "cuda")
    q = batch.quantize(on_gpu, torch.tensor(widths, dtype=torch.int32, device="cuda"), [3, 4, 5, 6])
    outs = [torch.empty_like(x) for x in on_gpu]
    batch.dequantize(q, outs)
    for x, bits, seed, out in zip(on_gpu, widths, [3, 4, 5, 6], outs):
        alone = ops.op_dequantize(ops.op_quantize(x, bits, seed, rng_stream="fast"), x.shape)
        assert torch.equal(out.view(torch.int16), alone.view(torch.int16)), bits
