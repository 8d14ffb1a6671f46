"""The plan's map from blocks to tensors on either side of the number of tensors whose first blocks fit in LDS, and the packed
offsets over several rounds of its first workgroup, against the same counted on the host."""
import numpy as np
import pytest
import torch

from gact.batched import GROUPS_PER_BLOCK, BatchedQuantizer
from gact.cpp_extension import _abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 255, 256, 257, 2047, 2048, 2049])
def test_plan_equals_the_host_count(count):
    rng = np.random.default_rng(count)
    sizes = [int(n) for n in rng.choice([1, 256, 32768, 32769, 100000, 300000], count)]
    widths = [int(b) for b in rng.choice([1, 2, 4, 8], count)]
    batch = BatchedQuantizer(sizes, [torch.float16] * count, "cuda")
    memory = torch.zeros(64, dtype=torch.float16, device="cuda")
    arr = (_abi.BatchEntry * count)()
    for e, n, first, stats in zip(arr, sizes, batch.first_blocks, batch.stats_offsets):
        e.x, e.numel, e.dtype, e.first_block, e.stats_offset = memory.data_ptr(), n, _abi.F16, first, stats
    table = torch.frombuffer(bytearray(bytes(arr)), dtype=torch.uint8).cuda()
    ws = batch.new_workspace()
    bits = torch.tensor(widths, dtype=torch.int32, device="cuda")
    batch._launch_plan(table, bits, torch.empty(batch.arena_bytes_worst_case(), dtype=torch.uint8, device="cuda"), ws)
    spans = [(_abi.lib().gact_packed_bytes(b, -(-n // 256), 1, 256) + 255) // 256 * 256 for n, b in zip(sizes, widths)]
    assert ws[:16].view(torch.int64).tolist() == [sum(spans), 1]
    offsets = table.cpu().numpy().view(np.int64).reshape(-1, 7)[:, 5]
    np.testing.assert_array_equal(offsets, np.cumsum([0] + spans[:-1]))
    blocks = [-(-(-(-n // 256)) // GROUPS_PER_BLOCK) for n in sizes]
    of = ws[256:256 + 4 * batch.total_blocks].view(torch.int32).cpu().numpy()
    np.testing.assert_array_equal(of, np.repeat(np.arange(count), blocks))
