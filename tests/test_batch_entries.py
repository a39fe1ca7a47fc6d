"""Uneven batches: how long queue entries of the small class are and which stores it
uses, on both sides of the rules (no GPU), and parity of a list of short lines,
the one that stores plainly (rel-L2 vs the oracle, FP32 2e-7 log2 N, FP64
1e-14 log2 N)."""
import numpy as np
import pytest

import fftz
from gpu_util import rand_c, to_dev, tol
from oracle import oracle as O


def packed(lengths_and_batches):
    items, off = [], 0
    for n, b in lengths_and_batches:
        items.append((n, b, off, off))
        off += n * b
    return items, off


def small(items, prec):
    return fftz.batch_plan_json(items, prec)["classes"][0]


@pytest.mark.parametrize("prec", ["f", "d"])
def test_entries_follow_the_number_of_workgroups(prec):
    # items of 4096 points: one entry each where they keep the resident workgroups busy
    assert len(small(packed([(64, 64)] * 2000)[0], prec)["tiles"]) == 2000
    # too few of them: entries of 16 KiB, or one round of 32 lines
    assert len(small(packed([(64, 64)] * 200)[0], prec)["tiles"]) == 400
    # never beyond 4096 points, whatever the number
    assert len(small(packed([(64, 256)] * 2000)[0], prec)["tiles"]) == 8000


def test_stores():
    assert small(packed([(20, 50)] * 30)[0], "f")["nt"] == 0
    assert small(packed([(100, 5)] * 30)[0], "d")["nt"] == 0   # 1600 bytes a line
    assert small(packed([(200, 5)] * 30)[0], "d")["nt"] == 1   # 3200
    assert small(packed([(20, 50)] * 10 + [(2000, 20)] * 10)[0], "f")["nt"] == 1
    for c in fftz.batch_plan_json(packed([(20, 50), (8000, 1), (16384, 1)])[0], "f")["classes"][1:]:
        assert c["nt"] == 1 and len(c["tiles"]) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("direction", [0, 1])
def test_short_lines(torch_gpu, prec, direction):
    torch = torch_gpu
    items, total = packed([(1, 7), (2, 9), (13, 5), (16, 33), (17, 3), (24, 40), (37, 11), (64, 70), (100, 3), (61, 20)])
    x = rand_c((total,), 3, prec)
    dx = to_dev(torch, x)
    dy = torch.full_like(dx, float("nan"))
    p = fftz.BatchPlan(items, prec, direction)
    assert small(items, prec)["nt"] == 0 and p.execute_io(dx, dy) == 0
    torch.cuda.synchronize()
    y = dy.cpu().numpy()
    p.destroy()
    for n, b, io, oo in items:
        ref = O.fft(x[io:io + n * b].reshape(b, n).astype(np.complex128), -1 if direction == 0 else 1)
        assert O.rel_l2(y[oo:oo + n * b], ref.reshape(-1)) <= tol(max(n, 2), prec), (n, b)
