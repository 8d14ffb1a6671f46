"""The operators' native host side against the Python path behind it: the same bits for every form of call both take, and
nothing taken (None, so that the Python path answers) that needs a copy, a mode's or transform's attention, or a refusal."""
import pickle

import pytest
import torch

from gact import ops
from gact.batched import BatchedQuantizer
from gact.conf import config
from gact.cpp_extension import _abi, minimax, quantization


class _NoNative:
    """Every function answers None: the operators take their Python path."""

    def __getattr__(self, name):
        return lambda *args: None


class _Recorder:
    """The native functions, and which of them gave an answer."""

    def __init__(self):
        self.answers = {}

    def __getattr__(self, name):
        def call(*args):
            out = getattr(_NATIVE, name)(*args)
            self.answers.setdefault(name, []).append(out is not None)
            return out
        return call


_NATIVE = _abi.native()


def _both(monkeypatch, call, function, answers=True):
    """What the call gives by the native function of that name - which answers, or leaves it to Python - and without it."""
    recorder = _Recorder()
    with monkeypatch.context() as m:
        m.setattr(_abi, "native", lambda: recorder)
        taken = call()
    assert recorder.answers[function] == [answers]
    with monkeypatch.context() as m:
        m.setattr(_abi, "native", lambda: _NoNative())
        general = call()
    return taken, general


def _equal(a, b):
    if isinstance(a, torch.Tensor):
        return a.shape == b.shape and a.stride() == b.stride() and a.dtype == b.dtype and torch.equal(a, b)
    if isinstance(a, (list, tuple)):
        return len(a) == len(b) and all(_equal(x, y) for x, y in zip(a, b))
    return a == b


def _written(q, numel, bits, group):
    """Without the packed tensor's last byte, which nothing writes."""
    n = -(-(-(-numel // group)) // (8 // bits)) * group
    return [q[0][:n], q[1], q[2], q[3], q[0].numel()]


def test_arguments_that_are_not_ordinary_are_left_to_python():
    native = _abi.native()
    cpu = torch.zeros(4, 256)
    assert native.quantize(cpu, 4, 0, 0, 256) is None
    assert native.quantize([1.0], 4, 0, 0, 256) is None
    assert native.quantize(cpu, 4, 0) is None
    assert native.dequantize(torch.zeros(9, dtype=torch.int8), (4,), 4, cpu, cpu, 256) is None
    assert native.minimax(cpu) is None
    assert native.pack(cpu, cpu, cpu, 4, 0, 0) is None
    assert native.unpack(cpu, 4, cpu, cpu, 4, 1, 256) is None
    assert native.mask_pack(cpu.to(torch.uint8)) is None
    assert native.mask_unpack(cpu.to(torch.int32), 32) is None
    assert native.batch_table(b"", [], []) is None


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape,layout", [((1, 1), "dense"), ((255,), "dense"), ((3, 7, 171), "dense"), ((2, 16, 20, 20), "channels_last"),
                                          ((2, 49, 4, 32), "heads"), ((2, 49, 3, 10), "heads"), ((7, 600), "sliced")])
def test_round_trips_equal_the_python_path(monkeypatch, dtype, shape, layout):
    x = torch.randn(shape, device="cuda").to(dtype)
    if layout == "channels_last":
        x = x.contiguous(memory_format=torch.channels_last)
    elif layout == "heads":
        x = x.permute(0, 2, 1, 3)
    elif layout == "sliced":
        x = x.flatten()[1:]     # not aligned
    for bits in (1, 2, 4, 8):
        for stream in ("fast", "deterministic", "reference"):
            q, want = _both(monkeypatch, lambda: ops.op_quantize(x, bits, -5, rng_stream=stream), "quantize", layout != "sliced")
            assert _equal(_written(q, x.numel(), bits, 256), _written(want, x.numel(), bits, 256)), (bits, stream)
            assert _equal(*_both(monkeypatch, lambda: ops.op_dequantize(q, x.shape), "dequantize")), (bits, stream)


@pytest.mark.gpu
@pytest.mark.parametrize("group,stream", [(256, "fast"), (256, "reference"), (128, "fast")])
def test_layouts_without_a_kernel_are_copied_in_the_native_call(group, stream):
    for x in (torch.randn(4, 3, 16, 16, device="cuda").contiguous(memory_format=torch.channels_last),
              torch.randn(33, 50, device="cuda")[:, 3:20], torch.randn(6, 40, device="cuda").t()[::2]):
        assert not x.is_contiguous()
        mode = _abi.NOISE_MODES[stream]
        p, q = (_abi.native().quantize(t, 4, 7, mode, group) for t in (x, x.contiguous()))
        assert _equal(_written([p[0], 4, p[1], p[2]], x.numel(), 4, group), _written([q[0], 4, q[1], q[2]], x.numel(), 4, group))


@pytest.mark.gpu
@pytest.mark.parametrize("group", [64, 96, 128, 256, 512])
def test_group_sizes_and_extension_calls_equal_the_python_path(monkeypatch, group):
    monkeypatch.setattr(config, "group_size", group)
    x = torch.randn(5, group * 3 // 2, device="cuda")
    q, want = _both(monkeypatch, lambda: ops.op_quantize(x, 2, 3), "quantize", group != 96)
    assert _equal(_written(q, x.numel(), 2, group), _written(want, x.numel(), 2, group))
    assert _equal(*_both(monkeypatch, lambda: ops.op_dequantize(q, x.shape), "dequantize", group != 96))
    rows = torch.randn(6, group, device="cuda", dtype=torch.float16)
    mn, mx = minimax.minimax(rows)
    assert _equal(*_both(monkeypatch, lambda: minimax.minimax(rows), "minimax"))
    args = (rows.view(3, 2, group), mn.view(3, 2, 1), mx.view(3, 2, 1), 4, True, 9)
    (codes, scale), want = _both(monkeypatch, lambda: quantization.pack_single_precision(*args), "pack")
    assert _equal([codes[:-1], scale], [want[0][:-1], want[1]])
    assert _equal(*_both(monkeypatch, lambda: quantization.unpack_single_precision(codes, 4, scale, args[1], 3, 2, group), "unpack"))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 31, 512, 5000])
def test_masks_equal_the_python_path(monkeypatch, n):
    x = (torch.rand(n, device="cuda") < 0.5).to(torch.uint8)
    q, want = _both(monkeypatch, lambda: ops.op_quantize_mask(x), "mask_pack")
    assert _equal(q, want)
    assert _equal(*_both(monkeypatch, lambda: ops.op_dequantize_mask(q), "mask_unpack"))


@pytest.mark.gpu
def test_calls_that_are_not_ordinary_are_left_to_python():
    native = _abi.native()
    x = torch.randn(4, 256, device="cuda")

    class Sub(torch.Tensor):
        pass

    from torch.utils._python_dispatch import TorchDispatchMode

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    ok = (x, 4, 0, _abi.NOISE_FAST, 256)
    assert native.quantize(*ok) is not None
    for i, bad in ((0, x.as_subclass(Sub)), (0, x[:0]), (0, x.double()), (0, x.flatten()[1:]), (1, True), (1, 3), (1, 4.0), (2, 1 << 31),
                   (2, True), (3, -1), (3, _abi.NOISE_INJECT), (4, 96)):
        assert native.quantize(*(bad if k == i else a for k, a in enumerate(ok))) is None, (i, bad)
    with Watch():
        assert native.quantize(*ok) is None
    seen = []
    torch.vmap(lambda row: (seen.append(native.quantize(row, *ok[1:])), row)[1])(x)
    assert seen == [None]
    q = ops.op_quantize(x, 4, 0)
    for shape in ((4, 300), (4, -256), (0, 256), [4, 256], (1 << 40, 1 << 40)):
        assert native.dequantize(q[0], shape, 4, q[2], q[3], 256) is None, shape
    assert native.dequantize(q[0], x.shape, 4, q[2].half(), q[3], 256) is None


@pytest.mark.gpu
def test_batched_tables_and_verdicts(monkeypatch):
    xs = [torch.randn(n, device="cuda").to(dt) for n, dt in ((300, torch.float32), (70000, torch.float16), (256, torch.bfloat16))]
    batch = BatchedQuantizer([x.numel() for x in xs], [x.dtype for x in xs], "cuda")
    bits = torch.tensor([1, 4, 8], dtype=torch.int32, device="cuda")
    assert _equal(*_both(monkeypatch, lambda: batch._table(xs, [1, -2, 1 << 40]), "batch_table"))
    outs = {}
    side = torch.cuda.Stream()
    for name in ("here", "elsewhere"):
        with torch.cuda.stream(torch.cuda.current_stream() if name == "here" else side):
            torch.cuda.current_stream().wait_stream(torch.cuda.default_stream())
            outs[name] = batch.dequantize(batch.quantize(xs, bits, [4, 5, 6]))
    torch.cuda.synchronize()
    assert _equal(outs["here"], outs["elsewhere"])
    for x, b, seed, out in zip(xs, (1, 4, 8), (4, 5, 6), outs["here"]):
        assert torch.equal(out, ops.op_dequantize(ops.op_quantize(x, b, seed), x.shape))
    void = batch.quantize(xs, torch.tensor([1, 3, 8], dtype=torch.int32, device="cuda"), [4, 5, 6])
    with pytest.raises(RuntimeError, match="void"):
        batch.dequantize(void)
    with pytest.raises(RuntimeError, match="geometry"):
        batch.quantize(xs[::-1], bits, [4, 5, 6])
    assert "_verdict" not in void.__getstate__()
    assert pickle.loads(pickle.dumps(batch))._table(xs, [1, 2, 3]).numel() == 3 * 56


@pytest.mark.gpu
def test_results_are_allocated_as_torch_allocates_them():
    """Device, storage and inference marks of the native calls' results, and the byte nobody writes under deterministic mode, which
    fills new memory."""
    x = torch.randn(16, 512, device="cuda")
    q = ops.op_quantize(x, 4, 0)
    out = ops.op_dequantize(q, x.shape)
    for t in (q[0], q[2], q[3], out):
        like = torch.empty(t.shape, dtype=t.dtype, device="cuda")
        assert t.device == like.device and t.is_cuda and t.stride() == like.stride() and not t.requires_grad
        assert t.untyped_storage().nbytes() == like.untyped_storage().nbytes() and t.untyped_storage().resizable()
    assert not q[0].is_inference()
    with torch.inference_mode():
        assert ops.op_quantize(x, 4, 0)[0].is_inference()
    before = torch.cuda.memory_allocated()
    kept = ops.op_quantize(x, 8, 0)[0]
    assert torch.cuda.memory_allocated() > before
    del kept
    torch.use_deterministic_algorithms(True)
    try:
        assert ops.op_quantize(x, 4, 0)[0][-1].item() == torch.empty(1, dtype=torch.int8, device="cuda").item()
    finally:
        torch.use_deterministic_algorithms(False)
