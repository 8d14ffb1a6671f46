"""The calls whose speed counts: saved activations compressed and restored through the public entry points.

A case is one round trip (compress, then restore) of what a training iteration saves - or, for the last kind, one whole
hooked training step.  `listed` holds the sizes this repository's tests and benchmark use, `draw` more of the same ranges.
Run from the root of the repository.
"""
import math
import os
import sys

import torch
import torch.nn as nn
import torch.nn.functional as F

_PACKAGE = os.path.abspath("gact-icml_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import gact  # noqa: E402
from gact import ops  # noqa: E402
from gact.batched import BatchedQuantizer  # noqa: E402
from gact.conf import config  # noqa: E402
from gact.controller import Controller  # noqa: E402
from gact.cpp_extension import calc_precision, minimax, quantization  # noqa: E402

_DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_SIZES = {"f32": 4, "f16": 2, "bf16": 2}


def _tensor(name, shape, dtype, bits, stream="fast", data="randn", layout="contiguous", group=256):
    return {"name": name, "kind": "tensor", "shape": shape, "dtype": dtype, "bits": bits, "stream": stream, "data": data,
            "layout": layout, "group": group}


def listed():
    return [
        # the input of a small classifier's linear layer: a call that is all latency, as every saved tensor of a small
        # model is
        _tensor("small_f32_4bit", "16x512", "f32", 4),
        # the activation of an early convolution of a ResNet-50 at batch 128, after its ReLU: the largest single tensors
        _tensor("conv_f32_4bit", "128x256x56x56", "f32", 4, data="relu"),
        # hidden states of a BERT-large layer, 8 bit (optimisation level L1.1)
        _tensor("hidden_f16_8bit", "16384x1024", "f16", 8),
        # GELU inputs of the same layer as mixed-precision training on this GPU holds them
        _tensor("gelu_bf16_4bit", "16384x4096", "bf16", 4),
        # attention probabilities, 2 bit, with the noise stream of the reference (runs that have to reproduce it)
        _tensor("probs_f16_2bit_reference", "32x16x512x512", "f16", 2, stream="reference", data="softmax"),
        # node features of a graph network, 60 % zeros, 1 bit: a number of groups that 8 does not divide
        _tensor("gcn_f32_1bit", "169343x256", "f32", 1, data="relu60"),
        # config.group_size other than the default: finer groups for hidden states at 4 bit
        _tensor("groups128_f16_4bit", "16384x1024", "f16", 4, group=128),
        # a convolution's activation in the memory format half-precision convolutional networks are trained in
        _tensor("channels_last_f16_4bit", "64x256x56x56", "f16", 4, data="relu", layout="channels_last"),
        # the three extension calls on their own, as code written against the reference's extension makes them
        {"name": "extension_f32_2bit", "kind": "extension", "rows": 16384, "dtype": "f32", "bits": 2, "stream": "deterministic"},
        # dropout masks of attention probabilities, one byte per element, to bits and back
        {"name": "dropout_mask", "kind": "mask", "shape": "32x16x512x512", "keep": 0.9},
        # every saved tensor of a Swin-Tiny-like model in one batch: widths allocated on the GPU under a budget of 2 bits
        # per element, then one mixed-width compression and one restoration
        {"name": "batched_f16_mixed", "kind": "batched", "tensors": 120, "batch": 128, "dtype": "f16", "budget": 2.0},
        # one training step (forward, backward) of a small two-layer encoder under the hooks at level L1
        {"name": "train_encoder_f32_4bit", "kind": "train", "layers": 2, "hidden": 128, "heads": 4, "seq": 64, "batch": 16,
         "dtype": "f32", "level": "L1"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tensor", "tensor", "tensor", "reference", "group", "strided", "extension", "mask", "batched", "train"])
    dtype, bits = rng.choice(["f32", "f16", "bf16"]), rng.choice([1, 2, 4, 8])
    if kind in ("tensor", "reference"):
        cols = rng.choice([10, 64, 100, 197, 256, 512, 768, 1000, 1024, 3072, rng.randint(3, 4096)])
        rows = max(1, _log_int(rng, 1 << 10, 1 << 27) // cols)
        stream = "reference" if kind == "reference" else rng.choice(["fast", "fast", "fast", "deterministic"])
        return _unnamed(_tensor("", "%dx%d" % (rows, cols), dtype, bits, stream, rng.choice(["randn", "relu", "relu60", "softmax"])))
    if kind == "group":
        cols = rng.choice([64, 100, 768, 1024, rng.randint(3, 4096)])
        rows = max(1, _log_int(rng, 1 << 10, 1 << 26) // cols)
        return _unnamed(_tensor("", "%dx%d" % (rows, cols), rng.choice(["f32", "f16"]), bits, "fast", rng.choice(["randn", "relu"]),
                                group=rng.choice([64, 128, 512])))
    if kind == "strided":
        if rng.random() < 0.5:      # attention heads: [batch, seq, heads, width] seen as [batch, heads, seq, width]
            heads, width, seq = rng.choice([4, 12, 16]), rng.choice([32, 64, 80, 128]), rng.choice([49, 64, 197, 512, rng.randint(16, 1024)])
            batch = max(1, _log_int(rng, 1 << 12, 1 << 25) // (heads * width * seq))
            return _unnamed(_tensor("", "%dx%dx%dx%d" % (batch, heads, seq, width), dtype, bits, "fast", "randn", "heads"))
        channels, side = rng.choice([3, 16, 64, 96, 256, 512]), rng.choice([7, 14, 28, 32, 56, rng.randint(5, 64)])
        batch = max(1, _log_int(rng, 1 << 12, 1 << 26) // (channels * side * side))
        return _unnamed(_tensor("", "%dx%dx%dx%d" % (batch, channels, side, side), dtype, bits, "fast", "relu", "channels_last"))
    if kind == "extension":
        return {"kind": "extension", "rows": _log_int(rng, 16, 1 << 18), "dtype": rng.choice(["f32", "f16"]), "bits": bits,
                "stream": rng.choice(["fast", "deterministic"])}
    if kind == "mask":
        cols = rng.choice([64, 197, 512, 768, rng.randint(3, 4096)])
        return {"kind": "mask", "shape": "%dx%d" % (max(1, _log_int(rng, 1 << 12, 1 << 27) // cols), cols), "keep": rng.choice([0.5, 0.8, 0.9])}
    if kind == "batched":
        return {"kind": "batched", "tensors": rng.randint(12, 160), "batch": _log_int(rng, 1, 48), "dtype": dtype,
                "budget": rng.choice([2.0, 3.0, 4.0])}
    hidden, heads = rng.choice([(64, 2), (128, 4), (256, 4), (384, 6)])
    return {"kind": "train", "layers": rng.randint(1, 3), "hidden": hidden, "heads": heads, "seq": rng.choice([16, 49, 64, 100, 128]),
            "batch": _log_int(rng, 2, 32), "dtype": "f32", "level": rng.choice(["L1", "L1.1", "L1.2"])}


def _unnamed(case):
    del case["name"]
    return case


def _shape(case):
    return tuple(int(d) for d in case["shape"].split("x"))


def _values(shape, dtype, data, gen):
    x = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
    if data == "relu":
        x = torch.relu_(x)
    elif data == "relu60":
        x = torch.relu_(x.sub_(0.2533))     # P(N(0,1) < 0.2533) = 0.6
    elif data == "softmax":
        x = torch.softmax(x, dim=-1)
    return x.to(_DTYPES[dtype])


def _swin_shapes(case):
    """Token maps of the four stages of a Swin-Tiny-like model, in its proportions, earliest first."""
    b, n = case["batch"], case["tensors"]
    stages = [(b, 3136, 96), (b, 784, 192), (b, 196, 384), (b, 49, 768)]
    ends = (n // 6, n // 3, n - n // 6, n)
    return [stages[sum(i >= e for e in ends)] for i in range(n)]


class _Encoder(nn.Module):
    """Post-norm transformer encoder with written-out attention, then a classifier over the first token."""

    def __init__(self, layers, hidden, heads):
        super().__init__()
        self.heads = heads
        self.blocks = nn.ModuleList(nn.ModuleDict({
            "qkv": nn.Linear(hidden, 3 * hidden), "proj": nn.Linear(hidden, hidden), "norm1": nn.LayerNorm(hidden),
            "up": nn.Linear(hidden, 4 * hidden), "down": nn.Linear(4 * hidden, hidden), "norm2": nn.LayerNorm(hidden),
        }) for _ in range(layers))
        self.classifier = nn.Linear(hidden, 2)

    def forward(self, x):
        b, s, h = x.shape
        for blk in self.blocks:
            q, k, v = blk["qkv"](x).view(b, s, 3, self.heads, h // self.heads).permute(2, 0, 3, 1, 4)
            probs = torch.softmax(torch.matmul(q, k.transpose(-1, -2)) / math.sqrt(h // self.heads), dim=-1)
            x = blk["norm1"](x + blk["proj"](torch.matmul(probs, v).transpose(1, 2).reshape(b, s, h)))
            x = blk["norm2"](x + blk["down"](F.gelu(blk["up"](x))))
        return self.classifier(x[:, 0])


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "tensor":
        shape = _shape(case)
        if case["layout"] == "heads":
            b, h, s, d = shape
            x = _values((b, s, h, d), case["dtype"], case["data"], gen).permute(0, 2, 1, 3)
        elif case["layout"] == "channels_last":
            x = _values(shape, case["dtype"], case["data"], gen).contiguous(memory_format=torch.channels_last)
        else:
            x = _values(shape, case["dtype"], case["data"], gen)
        return {"case": case, "x": x, "seed": seed % 100003}
    if kind == "extension":
        return {"case": case, "x": _values((case["rows"], 256), case["dtype"], "randn", gen), "seed": seed % 100003}
    if kind == "mask":
        x = (torch.rand(_shape(case), generator=gen, device="cuda") < case["keep"]).to(torch.uint8)
        return {"case": case, "x": x}
    if kind == "batched":
        shapes = _swin_shapes(case)
        dtype = _DTYPES[case["dtype"]]
        numels = [math.prod(s) for s in shapes]
        xs = [_values(s, case["dtype"], "randn", gen) for s in shapes]
        # restored tensors live side by side in one buffer
        flat = torch.empty(sum(numels), dtype=dtype, device="cuda")
        outs = [o.view(s) for o, s in zip(flat.split(numels), shapes)]
        total = sum(numels)
        return {"case": case, "xs": xs, "flat": flat, "outs": outs, "batch": BatchedQuantizer(numels, [dtype] * len(xs), "cuda"),
                "sensitivity": torch.exp(2.0 * torch.randn(len(xs), generator=gen, device="cuda")),
                "numels": torch.tensor(numels, dtype=torch.int64, device="cuda"), "target": case["budget"] * total,
                "seeds": [seed % 100003 + i for i in range(len(xs))]}
    with torch.random.fork_rng(devices=["cuda"]):
        torch.manual_seed(seed)
        model = _Encoder(case["layers"], case["hidden"], case["heads"]).cuda().to(_DTYPES[case["dtype"]])
    shape = (case["batch"], case["seq"], case["hidden"])
    x = _values(shape, case["dtype"], "randn", gen).requires_grad_()
    labels = torch.randint(0, 2, (case["batch"],), generator=gen, device="cuda")
    gact.set_optimization_level(case["level"])
    return {"case": case, "model": model, "x": x, "labels": labels, "controller": Controller(model)}


def _codes(q_input, numel, bits, group):
    """The packed bytes that carry codes; the tensor's last byte is never written, here as in the reference."""
    per_byte = 8 // bits
    n_groups = -(-numel // group)
    return q_input[: -(-n_groups // per_byte) * group]


def _run_tensor(s):
    case, x = s["case"], s["x"]
    kept = config.group_size
    config.group_size = case["group"]
    try:
        q = ops.op_quantize(x, case["bits"], s["seed"], rng_stream=case["stream"])
        out = ops.op_dequantize(q, x.shape)
    finally:
        config.group_size = kept
    return {"codes": _codes(q[0], x.numel(), case["bits"], case["group"]), "scale": q[2], "min": q[3], "restored": out}


def _run_extension(s):
    case, x = s["case"], s["x"]
    n = x.shape[0]
    mn, mx = minimax.minimax(x)
    codes, scale = quantization.pack_single_precision(x.view(n, 1, 256), mn.view(n, 1, 1), mx.view(n, 1, 1), case["bits"], True,
                                                      s["seed"], rng_stream=case["stream"])
    out = quantization.unpack_single_precision(codes, case["bits"], scale, mn.view(n, 1, 1), n, 1, 256)
    return {"codes": _codes(codes, x.numel(), case["bits"], 256), "scale": scale, "min": mn, "max": mx, "restored": out}


def _run_mask(s):
    q = ops.op_quantize_mask(s["x"])
    return {"bits": q[0], "restored": ops.op_dequantize_mask(q)}


def _run_batched(s):
    bits = torch.full((len(s["xs"]),), 8, dtype=torch.int32, device="cuda")
    calc_precision.calc_precision_device(bits, s["sensitivity"], s["numels"], s["target"])
    q = s["batch"].quantize(s["xs"], bits, s["seeds"], arena_bytes=s["batch"].arena_bytes_for_budget(s["target"]))
    s["batch"].dequantize(q, s["outs"])
    return {"widths": bits, "restored": s["flat"]}


def _run_train(s):
    model, x, controller = s["model"], s["x"], s["controller"]
    model.zero_grad(set_to_none=True)
    x.grad = None
    with controller:
        loss = F.cross_entropy(model(x).float(), s["labels"])
        loss.backward()
    controller.iterate(None)
    return {"loss": loss.detach(), "input": x.grad, "parameters": [p.grad for p in model.parameters()]}


_RUN = {"tensor": _run_tensor, "extension": _run_extension, "mask": _run_mask, "batched": _run_batched, "train": _run_train}


def run(state):
    return _RUN[state["case"]["kind"]](state)


def _round_trip_bytes(numel, esize, bits, group, scale_size=None):
    """Compress and restore: elements, codes, scale and minimum, in one direction and back."""
    n = -(-numel // group)
    per_byte = 8 // bits
    return 2 * (numel * esize + -(-n // per_byte) * group + n * (esize + (scale_size or esize)))


def work(case):
    kind = case["kind"]
    if kind == "tensor":
        scale_size = 4 if case["dtype"] == "bf16" else None
        return {"bytes": _round_trip_bytes(math.prod(_shape(case)), _SIZES[case["dtype"]], case["bits"], case["group"], scale_size), "flops": 0}
    if kind == "extension":
        # minimax reads the elements, pack reads them again (the calls are separate), unpack writes them
        es, n = _SIZES[case["dtype"]], case["rows"]
        return {"bytes": 3 * n * 256 * es + 2 * (n * 256 * case["bits"] // 8) + 7 * n * es, "flops": 0}
    if kind == "mask":
        n = math.prod(_shape(case))
        return {"bytes": 2 * (n + -(-n // 32) * 4), "flops": 0}
    if kind == "batched":
        # at the budget's average width
        numel = sum(math.prod(s) for s in _swin_shapes(case))
        es = _SIZES[case["dtype"]]
        return {"bytes": 2 * int(numel * (es + case["budget"] / 8 + (es + max(es, 4 if case["dtype"] == "bf16" else es)) / 256)), "flops": 0}
    # forward and backward matrix products; parameters and their gradients, and every saved activation written as codes
    # and read back
    t, h, l = case["batch"] * case["seq"], case["hidden"], case["layers"]
    weights = l * (12 * h * h + 13 * h) + 2 * h + 2
    return {"bytes": 4 * (2 * weights + 2 * t * h), "flops": 3 * 2 * l * (12 * t * h * h + 2 * t * case["seq"] * h)}


def tolerance(case):
    if case["kind"] != "train":
        # codes, widths and restored values follow the inputs and the seed bit for bit
        return "exact"
    # gradients through 32-bit sums whose order the matrix products choose; a sum that ends up on the other side of a rounding
    # boundary moves a stored code by a step.  Seen with the input moved by 1e-7 of itself: 7e-4 and 0.018 where a code moved,
    # 1e-6 where none did.
    return {"rel": 3e-3, "max": 0.07}
