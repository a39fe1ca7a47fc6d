"""Column passes: the tile each rule gives on both sides of its line (no GPU), and
parity of those tiles with numpy in FP64 (rel-L2, FP32 2e-7 log2 N, FP64 1e-14
log2 N)."""
import numpy as np
import pytest

import fftz
from gpu_util import rand_c, to_dev, tol
from oracle import oracle as O

# columns of L points: rows of n0 lines, images, precision -> lines per tile C, threads per line TL
TILES = [
    # a thread limit never leaves single lines at element stride
    (2800, 350, 1, "d", 2, 256), (2500, 800, 1, "d", 2, 128),
    # four complex128 lines where the LDS holds one such tile, unless many idle
    (1300, 1000, 1, "d", 4, 128), (1372, 10, 135, "d", 2, 128),
    # few lines: as many threads as the stages use; two lines a tile for long ones
    (1125, 514, 1, "f", 4, 256), (1125, 3000, 1, "f", 8, 64), (2187, 40, 1, "f", 2, 256), (144, 130, 1, "d", 4, 16),
    # the whole LDS for fixed complex128 kernels
    (1024, 64, 40, "d", 8, 64), (1024, 100, 20, "d", 4, 64), (1024, 41, 146, "d", 4, 64), (2048, 64, 4, "d", 4, 128),
    (2048, 100, 10, "d", 4, 128), (2048, 335, 1, "d", 2, 128), (2048, 16, 2, "d", 2, 128), (4096, 100, 1, "d", 2, 256),
    # fixed kernels keep a wavefront
    (64, 48, 1, "d", 16, 4), (64, 8, 1, "f", 8, 4), (128, 16, 2, "f", 8, 8)]


def geometry(L, n0, b):
    return [(L, n0, n0)], [(n0, 1, 1), (b, L * n0, L * n0)]


@pytest.mark.parametrize("L,n0,b,prec,C,TL", TILES)
def test_choice(L, n0, b, prec, C, TL):
    (ln,) = fftz.plan_json(*geometry(L, n0, b), prec)["launches"]
    in_col, out_col = 8, 16
    assert ln["flags"] & in_col and ln["flags"] & out_col
    assert (ln["C"], ln["TL"]) == (C, TL)


@pytest.mark.gpu
@pytest.mark.parametrize("L,n0,b,prec,C,TL", TILES)
def test_parity(torch_gpu, L, n0, b, prec, C, TL):
    torch = torch_gpu
    x = rand_c((b, L, n0), L + n0, prec)
    dx = to_dev(torch, x)
    dy = torch.full_like(dx, float("nan"))
    for direction in (0, 1):
        p = fftz.Plan(*geometry(L, n0, b), prec, direction, inp=dx, out=dy)
        assert p.execute() == 0
        ref = np.fft.fft(x.astype(np.complex128), axis=1) if direction == 0 else \
            np.fft.ifft(x.astype(np.complex128), axis=1) * L
        assert O.rel_l2(dy.cpu().numpy(), ref) <= tol(L, prec), p.info
        p.destroy()
