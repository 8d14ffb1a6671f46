"""The verdict of a batch's plan, which the plan's kernel writes to the host: it is there while the stream still has later work, waits for
earlier work, and may be dropped before the plan has run."""
import ctypes

import pytest
import torch

from gact.batched import BatchedQuantizer
from gact.cpp_extension import _abi

pytestmark = pytest.mark.gpu

LONG = 100_000_000      # cycles: 0.04 s at least


@pytest.fixture
def batch():
    sizes = [70001, 256, 40000]
    xs = [torch.randn(n, device="cuda") for n in sizes]
    made = BatchedQuantizer(sizes, [torch.float32] * 3, "cuda")
    made._on_gpu()
    bits = torch.tensor([1, 2, 4], dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    return made, xs, bits


def test_the_verdict_does_not_wait_for_later_work(batch):
    made, xs, bits = batch
    q = made.quantize(xs, bits, [1, 2, 3])
    torch.cuda._sleep(LONG)
    assert not isinstance(q._verdict, tuple)
    planned = q._planned()
    assert not torch.cuda.current_stream().query()
    assert planned == q.ok() and planned[0]
    void = made.quantize(xs, bits, [1, 2, 3], arena_bytes=256)
    assert void._planned() == (False, planned[1])


def test_the_verdict_waits_for_earlier_work(batch):
    made, xs, bits = batch
    side = torch.cuda.Stream()
    for stream in (torch.cuda.current_stream(), side):
        with torch.cuda.stream(stream):
            torch.cuda._sleep(LONG)
            q = made.quantize(xs, bits, [1, 2, 3])
            assert not stream.query()
            assert q._planned() == q.ok()


def test_an_error_that_nobody_has_read_outlasts_the_wait(batch):
    made, xs, bits = batch
    with open("/proc/self/maps") as maps:
        hip = ctypes.CDLL(next(line.split()[-1] for line in maps if "libamdhip64" in line))
    torch.cuda._sleep(LONG)
    q = made.quantize(xs, bits, [1, 2, 3])
    left = hip.hipSetDevice(torch.cuda.device_count() + 7)
    assert left != 0
    planned = q._planned()
    assert hip.hipGetLastError() == left and hip.hipGetLastError() == 0
    assert planned == q.ok() and planned[0]


def test_a_stream_that_torch_was_given(batch):
    """It may be gone before the wait: an event behind the plan says when it has run."""
    made, xs, bits = batch
    with open("/proc/self/maps") as maps:
        hip = ctypes.CDLL(next(line.split()[-1] for line in maps if "libamdhip64" in line))
    handle = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(handle)) == 0
    with torch.cuda.stream(torch.cuda.ExternalStream(handle.value)):
        for cycles in (0, LONG):
            torch.cuda._sleep(cycles)
            q = made.quantize(xs, bits, [1, 2, 3])
            torch.cuda._sleep(LONG)
            planned = q._planned()
            assert not torch.cuda.current_stream().query()
            assert planned == q.ok() and planned[0]
            made.dequantize(q)
        made.quantize(xs, bits, [1, 2, 3])


def test_verdicts_dropped_before_the_plan_has_run(batch):
    """Their words are not handed out again before: pinned memory taken meanwhile keeps its values."""
    made, xs, bits = batch
    cycles = LONG
    for _ in range(8):          # until the stream had more to do before the plans than the host took for what follows
        torch.cuda._sleep(cycles)
        for _ in range(30):
            made.quantize(xs, bits, [1, 2, 3])
        words = [torch.full((2,), -7, dtype=torch.int64).pin_memory() for _ in range(50)]
        under_way = not torch.cuda.current_stream().query()
        torch.cuda.synchronize()
        assert all(w.tolist() == [-7, -7] for w in words)
        if under_way:
            break
        cycles *= 2
    assert under_way
    q = made.quantize(xs, bits, [1, 2, 3])
    assert q._planned() == q.ok()


def test_words_of_dropped_verdicts_are_used_again(batch):
    """Pinned memory does not grow with the batches that nobody waits for."""
    made, xs, bits = batch

    def drop():
        torch.cuda._sleep(LONG)
        for _ in range(30):
            made.quantize(xs, bits, [1, 2, 3])
        torch.cuda.synchronize()
        made.quantize(xs, bits, [1, 2, 3])              # finds the others' words written
        torch.cuda.synchronize()
        return torch.cuda.host_memory_stats()["num_host_alloc"]

    first = drop()
    assert [drop() for _ in range(3)] == [first] * 3


def test_what_is_no_verdict_is_refused():
    for args in ((), (None,), (1, 2)):
        with pytest.raises((TypeError, ValueError)):
            _abi.native().verdict_wait(*args)
