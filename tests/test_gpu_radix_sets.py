"""GPU parity on either side of the rule that picks the pass kernel by the
radices of the line (powers of two; up to 8; up to 12; all), on rows, columns,
real-packed lines (pair radix up to 6 and above) and Bluestein lines.
Tolerance: rel-L2 vs the oracle, FP32 2e-7 log2 N, FP64 1e-14 log2 N
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


@pytest.mark.parametrize("n", [2, 7, 8, 9, 12, 13, 16, 63, 100, 125, 143, 144, 512, 1372, 3234, 5040, 8190])
def test_rows_f64(torch_gpu, n):
    x = rand_c((19, n), n, "d")
    for direction in (0, 1):
        y, info = run_c2c(torch_gpu, x, direction=direction)
        assert O.rel_l2(y, O.fft(x, -1 if direction == 0 else 1)) <= tol(n, "d"), info


@pytest.mark.parametrize("n", [6, 7, 8, 35, 36, 42, 49, 64, 75, 81, 125, 675, 1372])
def test_real_f64(torch_gpu, n):
    torch = torch_gpu
    for m in (2 * n, n):
        x = np.random.default_rng(m).standard_normal((5, m))
        dx = to_dev(torch, x)
        dy = torch.full((5, m // 2 + 1), float("nan"), dtype=torch.complex128, device="cuda")
        back = torch.full((5, m), float("nan"), dtype=torch.float64, device="cuda")
        p = fftz.Plan([(m, 1, 1)], [(5, m, m // 2 + 1)], "d", 0, fft_type=1, inp=dx, out=dy)
        q = fftz.Plan([(m, 1, 1)], [(5, m // 2 + 1, m)], "d", 1, fft_type=1, inp=dy, out=back)
        assert p.execute() == 0
        y = dy.cpu().numpy()
        assert q.execute() == 0
        assert O.rel_l2(y, np.fft.rfft(x)) <= tol(m, "d"), p.info
        assert O.rel_l2(back.cpu().numpy() / m + 0j, x + 0j) <= 2 * tol(m, "d"), q.info
        p.destroy()
        q.destroy()


@pytest.mark.parametrize("n,prec", [(37, "d"), (61, "f"), (101, "d"), (241, "f"), (601, "d"), (1009, "f"), (1277, "d")])
def test_bluestein(torch_gpu, n, prec):
    x = rand_c((7, n), n, prec)
    y, info = run_c2c(torch_gpu, x)
    assert O.rel_l2(y, O.fft(x.astype(np.complex128))) <= tol(4 * n, prec), info
