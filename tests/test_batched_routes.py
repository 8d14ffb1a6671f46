"""Which batches `BatchedQuantizer.dequantize` restores by the plan of their quantize call and which it plans again, without a GPU: the
launches and the native calls only write down that they were asked for."""
import pickle

import pytest
import torch

from gact.batched import BatchedPacked, BatchedQuantizer
from gact.cpp_extension import _abi


class _Nothing:
    def __enter__(self):
        return self

    def __exit__(self, *args):
        return False


class _Native:
    def __init__(self, routes):
        self.routes = routes

    def batch_dequantize(self, *args):
        self.routes.append("kept plan")
        return True


@pytest.fixture
def routes(monkeypatch):
    """What the dequantize calls of the test took, in order."""
    taken = []
    monkeypatch.setattr(torch.cuda, "device", lambda device: _Nothing())
    monkeypatch.setattr(_abi, "native", lambda: _Native(taken))
    monkeypatch.setattr(BatchedQuantizer, "_on_gpu", lambda self: torch.empty(0))
    monkeypatch.setattr(BatchedQuantizer, "_table", lambda self, *args, **kw: torch.empty(0))
    monkeypatch.setattr(BatchedQuantizer, "launch_dequantize", lambda self, *args: taken.append("own plan"))
    return taken


F32, F16 = torch.float32, torch.float16


def packed_by(batch):
    def memory(n):
        return torch.zeros(n, dtype=torch.uint8)

    return BatchedPacked(batch, memory(batch.arena_bytes_worst_case()), memory(batch.total_groups * 4), memory(batch.total_groups * 4),
                         memory(56 * batch.L), torch.ones(batch.L, dtype=torch.int32), memory(batch.workspace_bytes),
                         [torch.Size([n]) for n in batch.numels], list(batch.dtypes), list(range(batch.L)))


@pytest.mark.parametrize("numels,dtypes,same", [
    ([300, 70], [F32, F16], True),
    ([100, 70], [F32, F16], False),        # fewer elements in as many blocks: the table would write past the output
    ([300, 70], [F16, F16], False),        # half where the table holds float
    ([70, 300], [F16, F32], False),
    ([300], [F32], False),
])
def test_a_batch_of_another_quantizer(routes, numels, dtypes, same):
    """The plan is that of the quantizer that compressed; another one takes it only where it is the same tensor by tensor."""
    q = packed_by(BatchedQuantizer([300, 70], [F32, F16], "cpu"))
    outs = [torch.empty(n, dtype=d) for n, d in zip(numels, dtypes)]
    other = BatchedQuantizer(numels, dtypes, "cpu")
    other.dequantize(q, outs, check=False)
    pickle.loads(pickle.dumps(other)).dequantize(pickle.loads(pickle.dumps(q)), outs, check=False)
    q.owner.dequantize(q, check=False)
    q.owner = None      # a batch put together by hand
    other.dequantize(q, outs, check=False)
    assert routes == ["kept plan" if same else "own plan"] * 2 + ["kept plan", "own plan"]


def test_an_arena_cut_after_the_call(routes):
    """The plan vouches for the bytes there were when it was made; with fewer the next plan decides whether they are enough."""
    batch = BatchedQuantizer([300, 70], [F32, F16], "cpu")
    q = packed_by(batch)
    q.packed = torch.cat([q.packed, q.packed])      # a copy with room behind it
    batch.dequantize(q, check=False)
    q.packed = q.packed[:512].clone()
    batch.dequantize(q, check=False)
    batch.dequantize(pickle.loads(pickle.dumps(q)), check=False)
    older = packed_by(batch)
    del older._arena_bytes      # as unpickled from a file that does not say
    batch.dequantize(older, check=False)
    assert routes == ["kept plan", "own plan", "own plan", "own plan"]


@pytest.mark.parametrize("around", ["functionalize", "jvp", "fake"])
def test_the_geometry_is_not_made_inside_a_transform_or_a_mode(around, monkeypatch):
    """It is kept for later calls, so it must not be a wrapper that only means something there."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    batch = BatchedQuantizer([300], [F32], "cpu")
    batch.device = torch.device("meta")     # a copy to another device, which a transform wraps
    seen = []

    def inside(x):
        seen.append(batch._on_gpu())
        return x

    x = torch.ones(2)
    if around == "fake":
        with FakeTensorMode(allow_non_fake_inputs=True):
            inside(x)
    elif around == "functionalize":
        torch.func.functionalize(inside)(x)
    else:
        torch.func.jvp(inside, (x,), (x,))
    assert seen == [None] and batch._geometry is None
    assert batch._on_gpu() is batch._geometry and type(batch._geometry) is torch.Tensor
