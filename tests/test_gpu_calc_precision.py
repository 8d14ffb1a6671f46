"""The allocation on the GPU against the oracle where its search can go wrong: one candidate per thread, the sizes at which a thread
takes four and sixteen, tensors that start at different widths (1 among them), targets that a step meets exactly or just misses,
keys that share all but their last bits, sums over 2^32, no step needed, every step needed."""
import numpy as np
import pytest
import torch

import oracle
from gact.cpp_extension import calc_precision as ext

pytestmark = pytest.mark.gpu


def check(b, C, w, target):
    want = oracle.calc_precision(b, C, w, target)
    status = torch.full((1,), 99, dtype=torch.int32, device="cuda")
    got = ext.calc_precision_device(torch.from_numpy(b).cuda(), torch.from_numpy(C).cuda(), torch.from_numpy(w).cuda(), target, status)
    np.testing.assert_array_equal(got.cpu().numpy(), want, err_msg="L %d target %r" % (b.size, target))
    assert status.item() == 0


@pytest.mark.parametrize("L", [1, 2, 15, 16, 17, 255, 256, 257, 1023, 1024, 1025, 4095, 4096])
def test_search_equals_the_oracle(L):
    rng = np.random.default_rng(L)
    for spread in (0.0, 1e-6, 3.0):
        C = np.exp(rng.normal(0, spread, L)).astype(np.float32) if spread else np.full(L, 0.75, np.float32)
        C[rng.random(L) < 0.05] = 0.0
        for sizes in ("equal", "mixed", "large"):
            w = np.full(L, 4096, np.int64) if sizes == "equal" else (rng.integers(1, 60, L) * 256).astype(np.int64)
            if sizes == "large":
                w *= 1 << 24
            for widths in ((8,), (32,), (1, 2, 4, 8, 32)):
                b = rng.choice(widths, L).astype(np.int32)
                counted = float((b * w)[b > 1].sum())              # what the greedy counts before its first step
                least = float(w[b > 1].sum())                      # and after its last one
                for share in (0.0, 0.4, 1.0):
                    target = least + share * (counted - least)
                    check(b.copy(), C, w, target if share in (0.0, 1.0) else np.floor(target) + 0.5)


def test_targets_met_exactly_by_a_step():
    C = np.array([3.0, 1.0, 2.0], np.float32)
    w = np.full(3, 512, np.int64)
    for steps in range(10):                                        # 8 -> 4 -> 2 -> 1 three times
        full = 3 * 8 * 512
        for target in range(full, 3 * 512 - 1, -512):
            check(np.full(3, 8, np.int32), C, w, float(target))
            if target > 3 * 512:
                check(np.full(3, 8, np.int32), C, w, float(target) - 0.25)
        C = np.roll(C, 1) * np.float32(1.25)
