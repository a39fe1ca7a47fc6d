"""GPU parity of complex64 plain passes on either side of the rule that picks
the kernel by the radices of the line (pow2 only; none of 11, 13, 16; all), on
rows and on columns.  Tolerance: rel-L2 vs the oracle, FP32 2e-7 log2 N
(gpu_util.tol), as for every plain transform."""
import numpy as np
import pytest

import fftz
from gpu_util import rand_c, run_c2c, to_dev, tol
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 8, 9, 10, 11, 12, 16, 63, 100, 120, 143, 144, 160, 176, 1000, 1728, 1920, 6400])
def test_rows(torch_gpu, n):
    x = rand_c((37, n), n, "f")
    for direction in (0, 1):
        y, info = run_c2c(torch_gpu, x, direction=direction)
        assert O.rel_l2(y, O.fft(x.astype(np.complex128), -1 if direction == 0 else 1)) <= tol(n, "f"), info


@pytest.mark.parametrize("n0,n1", [(9, 16), (12, 35), (100, 33), (120, 96), (144, 5), (360, 77)])
def test_columns(torch_gpu, n0, n1):
    torch = torch_gpu
    x = rand_c((3, n0, n1), n0 * n1, "f")
    dx = to_dev(torch, x)
    dy = torch.full_like(dx, float("nan"))
    p = fftz.Plan([(n1, 1, 1), (n0, n1, n1)], [(3, n0 * n1, n0 * n1)], "f", 0, inp=dx, out=dy)
    assert p.execute() == 0
    ref = np.fft.fft2(x.astype(np.complex128))
    assert O.rel_l2(dy.cpu().numpy(), ref) <= tol(n0 * n1, "f"), p.info
    p.destroy()
