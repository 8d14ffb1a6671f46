"""The rules by which quantize of strided tensors chooses its kernel and the tile or strip it works on, taken from the library's source as
they stand there and built for the host: what the tests of those kernels check their shapes against."""
import ctypes
import functools
import os
import re
import subprocess
import tempfile

from conftest import ROOT

WRAP = """
extern "C" {
int takes(int size, int bits, int64_t numel, int64_t K) { return takes_strips(size, bits, numel, K); }
int tile(int size, int bits, int64_t numel, int64_t K) { return transposed_tile(size, bits, numel, K); }
int pay(int size, int bits, int64_t numel, int64_t M, int64_t K) { return tiles_pay(size, bits, numel, M, K, transposed_tile(size, bits, numel, K)); }
void cut(int bits, int64_t strips, int64_t K, int64_t* out) { const StripCut c = strip_cut(bits, strips, K); out[0] = c.gs; out[1] = c.segments; }
}
"""


@functools.lru_cache(maxsize=None)
def rules():
    with open(os.path.join(ROOT, "gact-icml_amd", "csrc", "gact_hip.hip")) as f:
        text = f.read()
    group = re.search(r"^#define GROUP \d+", text, re.M) or re.search(r"^.*\bGROUP = \d+;", text, re.M)
    start = text.index("inline bool takes_strips")
    end = text.index("\ntemplate", text.index("inline bool tiles_pay"))
    with tempfile.TemporaryDirectory() as place:
        out = os.path.join(place, "rules.so")
        source = "#include <cstddef>\n#include <cstdint>\n" + group.group(0) + "\n" + text[start:end] + WRAP
        subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-x", "c++", "-", "-o", out], input=source, text=True, check=True)
        lib = ctypes.CDLL(out)
    i64 = ctypes.c_int64
    lib.takes.argtypes = lib.tile.argtypes = [ctypes.c_int, ctypes.c_int, i64, i64]
    lib.pay.argtypes = [ctypes.c_int, ctypes.c_int, i64, i64, i64]
    lib.cut.argtypes = [ctypes.c_int, i64, i64, ctypes.POINTER(i64)]
    return lib


def strip_cut(size, bits, shape):
    """(groups of a channel per step, segments) of [batch, channels, pixels], or None where it is not worked in strips."""
    b, m, k = shape
    width = 16 // size
    numel = b * m * k
    if not rules().takes(size, bits, numel, k) or (m == width and bits < 8 and rules().pay(size, bits, numel, m, k)):
        return None
    out = (ctypes.c_int64 * 2)()
    rules().cut(bits, -(-m // (4 * width)) * b, k, out)
    return tuple(out)


def tile(size, bits, shape):
    """Elements of a tile, or None where the tensor is worked in strips or copied first."""
    b, m, k = shape
    if strip_cut(size, bits, shape) or not rules().pay(size, bits, b * m * k, m, k):
        return None
    return rules().tile(size, bits, b * m * k, k)
