"""What the operators' Python path refuses, copies and hands on, without a GPU: tensors in host memory that say they are on the
GPU, and a library that only writes down which entry point was called."""
import ctypes

import pytest
import torch

from gact import ops
from gact.batched import BatchedQuantizer
from gact.conf import config
from gact.cpp_extension import _abi, minimax, quantization


class _SaysGpu(torch.Tensor):
    is_cuda = property(lambda self: True)


class _Library:
    """Every entry point succeeds and is noted with its arguments."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            self.calls.append((name, args))
            return 0
        return call


@pytest.fixture
def library(monkeypatch):
    lib = _Library()
    _abi.native()       # the real one: it leaves tensors that are not plain GPU tensors to Python
    monkeypatch.setattr(_abi, "lib", lambda: lib)
    monkeypatch.setattr(_abi, "call_on", lambda device, fn, *args: fn(*args))
    monkeypatch.setattr(_abi, "stream_of", lambda t: 0)
    monkeypatch.setattr(ops, "_current_stream", lambda index: 0)
    monkeypatch.setattr(torch.cuda, "device", lambda device: _Nothing())
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    saved = config.group_size
    yield lib
    config.group_size = saved


class _Nothing:
    def __enter__(self):
        return self

    def __exit__(self, *args):
        return False


class _NoTables:
    def batch_table(self, *args):
        return None


def gpu(t):
    return t.as_subclass(_SaysGpu)


def _compressed(group, bits=4, groups=6):
    codes = gpu(torch.zeros(quantization.packed_numel(bits, groups, 1, group), dtype=torch.int8))
    return [codes, bits, gpu(torch.ones(groups, 1, 1)), gpu(torch.zeros(groups, 1, 1))]


@pytest.mark.parametrize("group", [64, 128, 256, 512])
def test_dequantize_takes_dense_gpu_memory_only(library, group):
    config.group_size = group
    shape = (6, group)
    ops.op_dequantize(_compressed(group), shape)
    assert len(library.calls) == 1
    n = _compressed(group)[0].numel()
    bad = [(0, torch.zeros(n, dtype=torch.int8), "data must be a CUDA tensor"),
           (0, gpu(torch.zeros(2 * n, dtype=torch.int8)[::2]), "data must be contiguous"),
           (0, gpu(torch.zeros(1, dtype=torch.int8).expand(n)), "data must be contiguous")]
    for i, name in ((2, "scale"), (3, "min")):
        bad += [(i, torch.ones(6, 1, 1), name + " must be a CUDA tensor"),
                (i, gpu(torch.ones(1, 1, 1).expand(6, 1, 1)), name + " must be contiguous"),
                (i, gpu(torch.ones(12, 1, 1)[::2]), name + " must be contiguous")]
        if group != 256:
            bad.append((i, gpu(torch.ones(6)), "dimension of %s" % name))
    for i, t, message in bad:
        q = _compressed(group)
        q[i] = t
        with pytest.raises(RuntimeError, match=message):
            ops.op_dequantize(q, shape)
    assert len(library.calls) == 1


def test_mask_is_dense_gpu_memory(library):
    for t, message in ((torch.zeros(4, dtype=torch.int32), "mask must be a CUDA tensor"),
                       (gpu(torch.zeros(8, dtype=torch.int32)[::2]), "mask must be contiguous"),
                       (gpu(torch.zeros(1, dtype=torch.int32).expand(4)), "mask must be contiguous")):
        with pytest.raises(RuntimeError, match=message):
            quantization.act_dequantize_dropout_mask(t, 128)
    assert not library.calls
    quantization.act_dequantize_dropout_mask(gpu(torch.zeros(4, dtype=torch.int32)), 128)
    assert len(library.calls) == 1


def _floats(address, n):
    return list((ctypes.c_float * n).from_address(address))


def _words(address, n):
    return list((ctypes.c_int32 * n).from_address(address))


def _negated(t):
    return gpu(torch._neg_view(-t))


@pytest.mark.parametrize("group", [128, 256])
def test_lazily_negated_views_are_resolved(library, group, monkeypatch):
    """A dense one is contiguous: what goes to the library is its values, not its memory, which holds them with the other sign."""
    config.group_size = group
    seen = []

    def entry(*indices):
        def call(*args):
            seen.append([_floats(args[i], n) for i, n in indices])
            return 0
        return call

    n = 2 * group
    x, stats = torch.arange(1.0, n + 1).view(2, group), torch.tensor([3.0, 5.0]).view(2, 1, 1)
    values, two = x.flatten().tolist(), [3.0, 5.0]
    library.gact_quantize = library.gact_quantize_groups = entry((0, n))
    ops.op_quantize(_negated(x), 4, 0)
    library.gact_dequantize = library.gact_dequantize_groups = entry((2, 2), (3, 2))
    q = _compressed(group, groups=2)
    ops.op_dequantize([q[0], 4, _negated(stats), _negated(stats)], (2, group))
    library.gact_minimax = entry((0, n))
    minimax.minimax(_negated(x))
    library.gact_pack = entry((0, n), (1, 2), (2, 2))
    quantization.pack_single_precision(_negated(x.view(2, 1, group)), _negated(stats), _negated(stats), 4, True, 0)
    library.gact_unpack = entry((2, 2), (3, 2))
    quantization.unpack_single_precision(q[0], 4, _negated(stats), _negated(stats), 2, 1, group)
    assert seen == [[values], [two, two], [values], [values, two, two], [two, two]]
    library.gact_batch_workspace_bytes = lambda *args: 4096
    batch = BatchedQuantizer([n], [torch.float32], "cpu")
    monkeypatch.setattr(_abi, "native", lambda: _NoTables())       # the native one asks for pinned memory first
    batch._table([gpu(x)], [0])
    with pytest.raises(RuntimeError, match="resolve_neg"):
        batch._table([_negated(x)], [0])


def test_lazily_negated_masks_are_resolved(library):
    seen = []
    library.gact_mask_pack = lambda x, n, *args: seen.append((ctypes.c_uint8 * n).from_address(x)[:]) or 0
    library.gact_mask_unpack = lambda x, n, *args: seen.append(_words(x, 2)) or 0
    ops.op_quantize_mask(gpu(torch._neg_view(torch.tensor([0, 255, 255, 0], dtype=torch.uint8))))
    ops.op_dequantize_mask([_negated(torch.tensor([5, 9], dtype=torch.int32)), (64,)])
    assert seen == [[0, 1, 1, 0], [5, 9]]


@pytest.mark.parametrize("group", [64, 128, 512])
def test_codes_and_noise_at_any_address(library, group):
    """The one-pass kernels are for 16-byte aligned memory: other codes take unpack, other noise is copied first."""
    config.group_size = group
    q = _compressed(group)
    for offset, entry in ((0, "gact_dequantize_groups"), (1, "gact_unpack"), (16, "gact_dequantize_groups")):
        buffer = torch.zeros(q[0].numel() + 16, dtype=torch.int8)
        assert buffer.data_ptr() % 16 == 0
        library.calls.clear()
        ops.op_dequantize([gpu(buffer[offset:offset + q[0].numel()])] + q[1:], (6, group))
        assert [name for name, _ in library.calls] == [entry], offset
    x, noise = gpu(torch.zeros(6, group)), gpu(torch.zeros(6 * group + 1))
    for part in (noise[:-1], noise[1:]):
        library.calls.clear()
        ops.op_quantize(x, 4, 1, noise=part)
        (name, args), = library.calls
        assert name == "gact_quantize_groups" and args[8] % 16 == 0


@pytest.mark.gpu
@pytest.mark.parametrize("group", [64, 128, 512])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16], ids=["f32", "f16"])
def test_codes_and_noise_at_any_address_on_the_gpu(group, dtype, monkeypatch):
    monkeypatch.setattr(config, "group_size", group)
    x = torch.randn(5 * group + 3, device="cuda").to(dtype)
    noise = torch.rand(6 * group + 1, device="cuda")
    for bits in (1, 2, 4, 8):
        p, q = ops.op_quantize(x, bits, 1, noise=noise[1:]), ops.op_quantize(x, bits, 1, noise=noise[1:].clone())
        want = ops.op_dequantize(q, x.shape)
        assert torch.equal(p[0][:-1], q[0][:-1])
        codes = torch.cat([q[0][:1], q[0]])[1:]
        assert codes.data_ptr() % 16 == 1
        assert torch.equal(ops.op_dequantize([codes] + q[1:], x.shape), want)


@pytest.mark.gpu
@pytest.mark.parametrize("group", [64, 128, 256, 512])
def test_strided_statistics_codes_and_masks_are_refused_on_the_gpu(group, monkeypatch):
    """The native calls leave them to Python, which raises; nothing is launched."""
    monkeypatch.setattr(config, "group_size", group)
    x = torch.randn(6, group, device="cuda")
    q = ops.op_quantize(x, 4, 1)
    native = _abi.native()
    assert native.dequantize(q[0], x.shape, 4, q[2], q[3], group) is not None
    bad = [(0, torch.cat([q[0], q[0]])[::2], "data"), (0, q[0][:1].expand(q[0].numel()), "data"), (0, q[0].cpu(), "data"),
           (2, torch.cat([q[2], q[2]])[::2], "scale"), (2, q[2][:1].expand(6, 1, 1), "scale"), (2, q[2].cpu(), "scale"),
           (3, torch.cat([q[3], q[3]])[::2], "min"), (3, q[3][:1].expand(6, 1, 1), "min"), (3, q[3].cpu(), "min")]
    for i, t, name in bad:
        args = [t if k == i else v for k, v in enumerate(q)]
        assert native.dequantize(args[0], x.shape, 4, args[2], args[3], group) is None, (i, name)
        with pytest.raises(RuntimeError, match=name + " must be"):
            ops.op_dequantize(args, x.shape)
    mask = torch.zeros(8, dtype=torch.int32, device="cuda")
    for t in (mask[::2], mask[:1].expand(4)):
        assert native.mask_unpack(t, 128) is None
        with pytest.raises(RuntimeError, match="mask must be contiguous"):
            quantization.act_dequantize_dropout_mask(t, 128)
