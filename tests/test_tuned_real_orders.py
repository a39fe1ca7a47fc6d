"""Tuned radix orders of real-packed passes: every order that the cache accepts is
the one the plan runs, whatever radix falls on the stage of mirrored butterfly
pairs (last forward, first backward), and the result is the transform.
Tolerance: rel-L2 vs the oracle, FP32 2e-7 log2 N, FP64 1e-14 log2 N, twice that
for the round trip."""
import numpy as np
import pytest

import fftz
from gpu_util import tol
from oracle import oracle as O

# half length, order: pair stages of radix 16, 12, 13, 11 and below in either direction
ORDERS = [(256, "16.16"), (192, "16.12"), (192, "12.16"), (4096, "16.16.16"), (144, "12.12"), (208, "16.13"),
          (132, "12.11"), (16, "16"), (12, "12"), (512, "2.16.16"), (64, "4.16"), (3072, "16.16.12")]


def entry(half, batch, prec, direction, order):
    n, p = 2 * half, 4 if prec == "f" else 8
    a, b = (n, half + 1) if direction == 0 else (half + 1, n)
    return f"p{p}:{1 + direction}:{direction}:0:0|{n},1,1;|{batch},{a},{b}; 0 0 0 0 r={half}:{order}\n"


@pytest.mark.parametrize("half,order", ORDERS)
@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("direction", [0, 1])
def test_order_is_used(half, order, prec, direction):
    fftz.tune_clear()
    try:
        assert fftz.tune_parse(entry(half, 5, prec, direction, order)) == 1
        n = 2 * half
        vec = (5, n, half + 1) if direction == 0 else (5, half + 1, n)
        ln = fftz.plan_json([(n, 1, 1)], [vec], prec, direction, fft_type=1)["launches"]
        assert len(ln) == 1 and ln[0]["radix"] == [int(r) for r in order.split(".")]
    finally:
        fftz.tune_clear()


@pytest.mark.gpu
@pytest.mark.parametrize("half,order", ORDERS)
@pytest.mark.parametrize("prec", ["f", "d"])
def test_parity(torch_gpu, half, order, prec):
    torch = torch_gpu
    n, b = 2 * half, 5
    x = np.random.default_rng(n).standard_normal((b, n)).astype(np.float32 if prec == "f" else np.float64)
    dx = torch.from_numpy(x).cuda()
    dy = torch.full((b, half + 1), float("nan"), dtype=torch.complex64 if prec == "f" else torch.complex128, device="cuda")
    back = torch.full_like(dx, float("nan"))
    fftz.tune_clear()
    try:
        assert fftz.tune_parse(entry(half, b, prec, 0, order) + entry(half, b, prec, 1, order)) == 2
        p = fftz.Plan([(n, 1, 1)], [(b, n, half + 1)], prec, 0, fft_type=1, inp=dx, out=dy)
        q = fftz.Plan([(n, 1, 1)], [(b, half + 1, n)], prec, 1, fft_type=1, inp=dy, out=back)
    finally:
        fftz.tune_clear()
    frag = "r=" + order.replace(".", "x")
    assert frag in p.info and frag in q.info
    assert p.execute() == 0 and q.execute() == 0
    ref = O.fft(x.astype(np.complex128))[:, :half + 1]
    assert O.rel_l2(dy.cpu().numpy(), ref) <= tol(n, prec), p.info
    assert O.rel_l2(back.cpu().numpy().astype(np.complex128) / n, x.astype(np.complex128)) <= 2 * tol(n, prec), q.info
    p.destroy()
    q.destroy()
