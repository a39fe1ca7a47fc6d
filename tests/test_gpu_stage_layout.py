"""GPU parity of the generic pass kernels at the sizes where their in-place
digit layout can go wrong: one to five stages, remainder rounds of the
butterfly loops, lines narrower and wider than a wavefront, ragged batches;
real-packed pair stages of every radix (odd and even butterfly counts, the
self-mirrored butterflies 0 and nbl/2, the radix-11 / 13 kernel); Bluestein
plans of two to four stages.  Tolerance: rel-L2 vs the oracle, FP32
2e-7 log2 N, FP64 1e-14 log2 N (gpu_util.tol), as for every plain transform."""
import numpy as np
import pytest

import fftz
from gpu_util import rand_c, run_c2c, to_dev, tol
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# stages: 1, 2 (odd x odd), 2 (16 x 2), 3, 3 (all 11 / 13), 4, 5; the longest single pass
LENGTHS = [(13, 257), (33, 65), (32, 129), (286, 31), (1183, 17), (1331, 9), (1200, 7), (2310, 5), (6561, 3),
           (8192, 3)]


@pytest.mark.parametrize("n,batch", LENGTHS + [(10010, 2), (15015, 2), (16384, 2)])
@pytest.mark.parametrize("direction", [0, 1])
def test_complex64(torch_gpu, n, batch, direction):
    x = rand_c((batch, n), n, "f")
    y, info = run_c2c(torch_gpu, x, direction=direction)
    assert O.rel_l2(y, O.fft(x.astype(np.complex128), -1 if direction == 0 else 1)) <= tol(n, "f"), info


@pytest.mark.parametrize("n,batch", LENGTHS + [(5005, 2)])
def test_complex128(torch_gpu, n, batch):
    x = rand_c((batch, n), n, "d")
    y, info = run_c2c(torch_gpu, x)
    assert O.rel_l2(y, O.fft(x)) <= tol(n, "d"), info


# n/2 = 1, one stage of each pair radix, pair stage with odd / even butterfly
# counts, default plans without a pair radix (16 x 16, 16 x 12, 16^3), 11s and 13s only
HALVES = [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 16, 22, 30, 35, 63, 99, 100, 121, 143, 192, 208, 256, 325, 1331,
          1800, 2197, 4096]


@pytest.mark.parametrize("half", HALVES)
@pytest.mark.parametrize("prec", ["f", "d"])
def test_real_packed(torch_gpu, half, prec):
    torch = torch_gpu
    n, b = 2 * half, 5
    rng = np.random.default_rng(n)
    x = rng.standard_normal((b, n)).astype(np.float32 if prec == "f" else np.float64)
    dx = to_dev(torch, x)
    ct = torch.complex64 if prec == "f" else torch.complex128
    dy = torch.full((b, half + 1), float("nan"), dtype=ct, device="cuda")
    back = torch.full((b, n), float("nan"), dtype=dx.dtype, device="cuda")
    p = fftz.Plan([(n, 1, 1)], [(b, n, half + 1)], prec, 0, fft_type=1, inp=dx, out=dy)
    q = fftz.Plan([(n, 1, 1)], [(b, half + 1, n)], prec, 1, fft_type=1, inp=dy, out=back)
    assert p.execute() == 0 and q.execute() == 0
    ref = O.fft(x.astype(np.complex128))[:, :half + 1]
    assert O.rel_l2(dy.cpu().numpy(), ref) <= tol(n, prec), p.info
    assert O.rel_l2(back.cpu().numpy().astype(np.complex128) / n, x.astype(np.complex128)) <= 2 * tol(n, prec), q.info
    p.destroy()
    q.destroy()


@pytest.mark.parametrize("n", [17, 67, 509, 1009, 2053, 4093, 8191])
@pytest.mark.parametrize("prec", ["f", "d"])
def test_bluestein(torch_gpu, n, prec):
    if prec == "d" and n > 4096:
        pytest.skip("multi-pass in complex128")
    x = rand_c((3, n), n, prec)
    for direction in (0, 1):
        y, info = run_c2c(torch_gpu, x, direction=direction)
        assert "bluestein" in info
        assert O.rel_l2(y, O.fft(x.astype(np.complex128), -1 if direction == 0 else 1)) <= tol(4 * n, prec), info
