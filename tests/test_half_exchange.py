"""Fixed column passes whose exchanges run through half the LDS: the choice on both
sides of its rules (no GPU), and parity with numpy in FP64 where it is taken
(rel-L2, FP32 2e-7 log2 N, FP64 1e-14 log2 N)."""
import numpy as np
import pytest

import fftz
from gpu_util import rand_c, to_dev, tol
from oracle import oracle as O


def geometry(L, n0, b):
    return [(L, n0, n0)], [(n0, 1, 1), (b, L * n0, L * n0)]


@pytest.mark.parametrize("prec,L,n0,images,split", [
    ("d", 256, 16, 512, 0), ("d", 256, 16, 1024, 1), ("d", 256, 100, 80, 1),   # more tiles than two a CU
    ("d", 256, 257, 127, 1), ("d", 256, 257, 255, 0),                          # ragged rows up to 128 MiB
    ("d", 256, 512, 128, 1), ("d", 256, 512, 256, 0),                          # whole rows up to 256 MiB
    ("d", 512, 512, 64, 0), ("f", 256, 512, 64, 0), ("f", 1024, 512, 64, 0),
    ("f", 512, 512, 64, 0), ("f", 512, 512, 128, 1), ("f", 512, 64, 1024, 0),  # from 256 MiB, not in short rows
    ("f", 512, 257, 300, 1), ("f", 512, 12, 341, 0)])
def test_choice(prec, L, n0, images, split):
    (ln,) = fftz.plan_json(*geometry(L, n0, images), prec)["launches"]
    assert ln["form"] == "fixed" and ln["split"] == split


@pytest.mark.gpu
@pytest.mark.parametrize("prec,L,n0,images", [("d", 256, 16, 544), ("d", 256, 100, 80), ("f", 512, 257, 260)])
def test_parity(torch_gpu, prec, L, n0, images):
    torch = torch_gpu
    x = rand_c((images, L, n0), n0, prec)
    dx = to_dev(torch, x)
    dy = torch.full_like(dx, float("nan"))
    p = fftz.Plan(*geometry(L, n0, images), prec, 1, inp=dx, out=dy)
    assert p.execute() == 0 and " split" in p.info
    y = dy.cpu().numpy()
    p.destroy()
    assert np.isfinite(y).all()
    some = [0, 1, images // 2, images - 1]
    ref = np.fft.ifft(x[some].astype(np.complex128), axis=1) * L
    assert O.rel_l2(y[some], ref) <= tol(L, prec)
