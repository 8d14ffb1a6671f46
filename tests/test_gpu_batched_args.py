"""A batch whose addresses and seeds travel in the plan's launch (up to 192 tensors) and one that is a tensor too long for it, against
the tensors one by one: codes, scales, minima, widths kept and restored values bit for bit, and the plan's header."""
import pickle
import random

import pytest
import torch

from gact import ops
from gact.batched import BatchedQuantizer
from gact.cpp_extension import _abi

pytestmark = pytest.mark.gpu


def make(count):
    rng = random.Random(count)
    g = torch.Generator(device="cuda").manual_seed(count)
    sizes = [rng.choice([1, 255, 256, 257, 2048, 32768, 32769, rng.randint(1, 100000)]) for _ in range(count)]
    dtypes = [rng.choice([torch.float32, torch.float16, torch.bfloat16]) for _ in range(count)]
    xs = [torch.randn(n, generator=g, device="cuda").to(d) for n, d in zip(sizes, dtypes)]
    widths = [rng.choice([1, 2, 4, 8]) for _ in range(count)]
    return xs, widths, [rng.randint(-5, 1 << 20) for _ in range(count)], BatchedQuantizer(sizes, dtypes, "cuda")


@pytest.mark.parametrize("count", [1, 63, 64, 65, 192, 193])     # a wave's share of the plan, its end, the longest, one more
def test_batch_equals_its_tensors(count):
    assert _abi.BATCH_ARGS == 192
    xs, widths, seeds, batch = make(count)
    bits = torch.tensor(widths, dtype=torch.int32, device="cuda")
    native = _abi.native().batch_quantize(batch._entry_bytes(), batch._on_gpu(), xs, seeds, bits,
                                          (batch.total_blocks, batch.total_groups, batch.workspace_bytes, batch.arena_bytes_worst_case(), _abi.NOISE_FAST,
                                           batch.dtype_mask)) if count <= 192 else None
    assert (native is not None) == (count <= 192)
    q = batch.quantize(xs, bits, seeds)
    bits.fill_(32)     # the widths are kept as they were
    outs = batch.dequantize(q)
    assert q.ok() == (True, q.ok()[1]) and q.workspace[16:48].view(torch.int64).tolist() == [widths.count(b) for b in (1, 2, 4, 8)]
    for i, x in enumerate(xs):
        want = ops.op_quantize(x, widths[i], seeds[i])
        codes, b, scale, mn = q.per_tensor(i)
        assert b == widths[i] and torch.equal(codes, want[0][: codes.numel()])
        assert torch.equal(scale, want[2]) and torch.equal(mn, want[3])
        assert torch.equal(outs[i], ops.op_dequantize(want, x.shape))
    later = pickle.loads(pickle.dumps(q))
    assert all(torch.equal(a, b) for a, b in zip(later.owner.dequantize(later), outs))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["f32", "f16", "bf16"])
def test_batches_of_one_type_whatever_is_said_of_it(dtype):
    """The launch of a batch of one type is shaped for it; told of any type it gives the same bytes."""
    g = torch.Generator(device="cuda").manual_seed(1)
    sizes = [70000, 513, 256 * 128 * 9, 3]
    xs = [torch.randn(n, generator=g, device="cuda").to(dtype) for n in sizes]
    batch = BatchedQuantizer(sizes, [dtype] * 4, "cuda")
    q = batch.quantize(xs, torch.tensor([1, 2, 4, 8], dtype=torch.int32, device="cuda"), [1, 2, 3, 4])
    outs = batch.dequantize(q)
    batch.dtype_mask = 7
    assert all(torch.equal(a, b) for a, b in zip(outs, batch.dequantize(q)))


def test_void_plans_and_dropped_batches():
    xs, widths, seeds, batch = make(40)
    bits = torch.tensor(widths, dtype=torch.int32, device="cuda")
    for _ in range(30):       # nobody waits for these
        batch.quantize(xs, bits, seeds)
    small = batch.quantize(xs, bits, seeds, arena_bytes=512)
    with pytest.raises(RuntimeError, match="void"):
        batch.dequantize(small)
    bad = bits.clone()
    bad[-1] = 32
    with pytest.raises(RuntimeError, match="void"):
        batch.dequantize(batch.quantize(xs, bad, seeds))
    with pytest.raises(RuntimeError, match="geometry"):
        batch.quantize([x[:1] for x in xs], bits, seeds)
    q = batch.quantize(xs, bits, seeds)
    assert q.ok()[0] and all(torch.equal(a, ops.op_dequantize(ops.op_quantize(x, b, s), x.shape))
                             for a, x, b, s in zip(batch.dequantize(q), xs, widths, seeds))


def test_outputs_of_the_caller():
    xs, widths, seeds, batch = make(33)
    q = batch.quantize(xs, torch.tensor(widths, dtype=torch.int32, device="cuda"), seeds)
    want = batch.dequantize(q)
    flat = torch.zeros(sum((x.numel() + 7) // 8 * 8 * x.element_size() for x in xs) + 16 * len(xs), dtype=torch.uint8, device="cuda")
    outs, at = [], 0
    for x in xs:      # side by side in one buffer, each on a 16-byte boundary
        outs.append(flat[at:at + x.numel() * x.element_size()].view(x.dtype))
        at += (x.numel() * x.element_size() + 15) // 16 * 16
    assert all(torch.equal(a, b) for a, b in zip(batch.dequantize(q, outs), want))
    with pytest.raises(RuntimeError, match="geometry"):
        batch.dequantize(q, outs[::-1])
    with pytest.raises(RuntimeError, match="aligned"):
        batch.dequantize(q, [flat[4:4 + x.numel() * x.element_size()].view(x.dtype) for x in xs])


def test_batches_on_streams_of_their_own():
    xs, widths, seeds, batch = make(20)
    bits = torch.tensor(widths, dtype=torch.int32, device="cuda")
    want = batch.dequantize(batch.quantize(xs, bits, seeds))
    torch.cuda.synchronize()
    outs = []
    streams = [torch.cuda.Stream() for _ in range(3)]
    for s in streams:
        with torch.cuda.stream(s):
            outs.append(batch.dequantize(batch.quantize(xs, bits, seeds)))
    del batch
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for o in outs for a, b in zip(o, want))


def test_a_batch_of_another_quantizer_fills_the_outputs_it_was_given():
    """Fewer elements in as many blocks: the beginning of the tensor, and not a byte behind it."""
    g = torch.Generator(device="cuda").manual_seed(2)
    xs = [torch.randn(n, generator=g, device="cuda") for n in (300, 40000)]
    q = BatchedQuantizer([300, 40000], [torch.float32] * 2, "cuda").quantize(xs, torch.tensor([4, 8], dtype=torch.int32, device="cuda"), [1, 2])
    want = q.owner.dequantize(q)
    flat = torch.full((64 * 1024,), 7.0, device="cuda")
    fewer = [flat[:100], flat[1024:1024 + 33000]]
    BatchedQuantizer([100, 33000], [torch.float32] * 2, "cuda").dequantize(q, fewer)
    assert torch.equal(fewer[0], want[0][:100]) and torch.equal(fewer[1], want[1][:33000])
    assert bool((flat[100:1024] == 7.0).all()) and bool((flat[1024 + 33000:] == 7.0).all())


def test_widths_written_over_after_the_call():
    """Codes end where the plan says: a tensor that its new width would take further is left as it is, the others keep to their codes."""
    sizes = [257, 256 * 128 * 3 + 5, 9]
    g = torch.Generator(device="cuda").manual_seed(3)
    xs = [torch.randn(n, generator=g, device="cuda") for n in sizes]
    batch = BatchedQuantizer(sizes, [torch.float32] * 3, "cuda")
    q = batch.quantize(xs, torch.tensor([1, 2, 4], dtype=torch.int32, device="cuda"), [1, 2, 3])
    want = batch.dequantize(q)
    for widths, untouched in [([1, 2, 4], []), ([1, 4, 4], [1]), ([8, 8, 8], [1]), ([1, 2, 8], []), ([2, 1, 32], [])]:
        q.bits.copy_(torch.tensor(widths, dtype=torch.int32))
        outs = batch.dequantize(q, [torch.full((n,), 7.0, device="cuda") for n in sizes])
        for i, (a, b) in enumerate(zip(outs, want)):
            assert bool((a == 7.0).all()) == (i in untouched), (widths, i)
            assert widths[i] != (1, 2, 4)[i] or torch.equal(a, b)


def test_a_batch_dropped_while_another_stream_waits_to_restore_it():
    """Nothing of it is handed out again before that stream has read it."""
    xs, widths, seeds, batch = make(24)
    bits = torch.tensor(widths, dtype=torch.int32, device="cuda")
    want = batch.dequantize(batch.quantize(xs, bits, seeds))
    q = batch.quantize(xs, bits, seeds)
    torch.cuda.synchronize()
    held = [q.packed, q.scale, q.min, q.table, q.workspace, q.bits]
    spans = [(t.data_ptr(), t.numel() * t.element_size()) for t in held]
    late = torch.cuda.Stream()
    with torch.cuda.stream(late):
        torch.cuda._sleep(100_000_000)      # 0.05 s at least
        outs = batch.dequantize(q)
    del held, q
    fresh = [torch.full((n,), 255, dtype=torch.uint8, device="cuda") for _, n in spans]
    assert not late.query()
    assert not any(t.data_ptr() < at + n and at < t.data_ptr() + t.numel() for t in fresh for at, n in spans)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(outs, want))


@pytest.mark.parametrize("blocks", [(1 << 12) - 1, 1 << 12, (12 << 10) - 1, 12 << 10])
def test_half_batches_where_another_kernel_takes_over(blocks):
    """On either side of the sizes from which fewer widths pack their codes as bytes: every width, ragged ends, a long tensor at each width
    below 8."""
    sizes = [1, 257, 32769, 100003] * 4
    long = (blocks - sum(-(-n // 32768) for n in sizes)) // 3
    ends = [long, long, blocks - sum(-(-n // 32768) for n in sizes) - 2 * long]
    sizes += [n * 32768 - 5 for n in ends]
    widths = [b for b in (1, 2, 4, 8) for _ in range(4)] + [1, 2, 4]
    g = torch.Generator(device="cuda").manual_seed(blocks)
    xs = [torch.randn(n, generator=g, device="cuda", dtype=torch.float16) for n in sizes]
    xs[2][5], xs[6][300], xs[10][7] = float("nan"), float("inf"), 60000.0
    batch = BatchedQuantizer(sizes, [torch.float16] * len(xs), "cuda")
    assert batch.total_blocks == blocks
    q = batch.quantize(xs, torch.tensor(widths, dtype=torch.int32, device="cuda"), list(range(len(xs))))
    for i, x in enumerate(xs):
        want = ops.op_quantize(x, widths[i], i)
        codes, b, scale, mn = q.per_tensor(i)
        assert b == widths[i] and torch.equal(codes, want[0][: codes.numel()]), i
        assert torch.equal(scale.view(torch.int16), want[2].view(torch.int16)) and torch.equal(mn.view(torch.int16), want[3].view(torch.int16))


@pytest.mark.parametrize("blocks", [(1 << 10) - 1, 1 << 10, (10 << 10) - 1, 10 << 10])
def test_float_batches_where_the_launch_of_dequantize_changes(blocks):
    """On either side of the sizes from which fewer workgroups share a CU: by the quantize call's plan and by one of the outputs' own."""
    sizes = [1, 257, 32769, 100003]
    sizes.append((blocks - sum(-(-n // 32768) for n in sizes)) * 32768 - 5)
    widths = [8, 4, 2, 1, 4]
    g = torch.Generator(device="cuda").manual_seed(blocks)
    xs = [torch.randn(n, generator=g, device="cuda") for n in sizes]
    batch = BatchedQuantizer(sizes, [torch.float32] * len(xs), "cuda")
    assert batch.total_blocks == blocks
    q = batch.quantize(xs, torch.tensor(widths, dtype=torch.int32, device="cuda"), list(range(len(xs))))
    outs = batch.dequantize(q)
    table, again = batch._table(xs, q.seeds), [x.clone() for x in xs]
    batch.launch_dequantize(table, q.bits, q.packed, q.scale, q.min, batch.new_workspace())      # over the inputs
    for i, x in enumerate(again):
        want = ops.op_dequantize(ops.op_quantize(x, widths[i], i), x.shape)
        assert torch.equal(outs[i], want) and torch.equal(xs[i], want), i
