"""Long transforms as two wide passes or three narrow ones: the planner's choice
on both sides of its line, and parity with the oracle (rel-L2, FP32 2e-7 log2 N,
FP64 1e-14 log2 N) where tiles hold 16 lines down to 4 and rows straddle
cache lines."""
import numpy as np
import pytest

import fftz
from gpu_util import rand_c, run_c2c, tol
from oracle import oracle as O


@pytest.mark.parametrize("n,batch,prec,passes", [
    (1 << 18, 2, "f", 2), (1 << 20, 8, "f", 2), (1 << 20, 16, "f", 3), (1 << 21, 1, "f", 2), (1 << 22, 1, "f", 3),
    (1000000, 16, "f", 2), (3 << 20, 1, "f", 3), (1 << 21, 1, "d", 2), (1 << 21, 8, "d", 3), (1 << 22, 1, "d", 3)])
def test_choice(n, batch, prec, passes):
    assert len(fftz.plan_json([(n, 1, 1)], [(batch, n, n)], prec)["launches"]) == passes


@pytest.mark.gpu
@pytest.mark.parametrize("n,batch,prec", [(1 << 18, 3, "f"), (1 << 19, 1, "f"), (1 << 20, 1, "f"), (1000000, 2, "f"),
                                          (412500, 2, "f"), (150579, 3, "f"), (1 << 18, 2, "d"), (1 << 21, 1, "d"),
                                          (340200, 1, "d")])
def test_parity(torch_gpu, n, batch, prec):
    x = rand_c((batch, n), n % 1009, prec)
    for direction in (0, 1):
        y, info = run_c2c(torch_gpu, x, direction=direction)
        assert "passes=2" in info
        assert O.rel_l2(y, O.fft(x.astype(np.complex128), -1 if direction == 0 else 1)) <= tol(n, prec), info
