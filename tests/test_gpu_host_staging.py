"""Host output buffers: a dense output is written whole, an output with gaps
keeps the caller's elements between the results (the library copies it in first
only then)."""
import numpy as np
import pytest

import fftz
from gpu_util import tol
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# (dims, vecs, elements of the output buffer): innermost first, strides in elements
DENSE = [([(64, 1, 1)], [(5, 64, 64)], 320),
         ([(12, 5, 5)], [(5, 1, 1)], 60),                              # interleaved batch
         ([(8, 1, 1), (6, 8, 8)], [(2, 48, 48), (3, 96, 96)], 288),
         ([(6, 1, 8), (8, 6, 1)], [(3, 48, 48)], 144)]                 # transposed output
GAPS = [([(64, 1, 1)], [(5, 64, 70)], 344),
        ([(12, 1, 2)], [(5, 12, 30)], 143),
        ([(8, 1, 1), (6, 8, 9)], [(2, 48, 60)], 113)]


@pytest.mark.parametrize("dims,vecs,size", DENSE + GAPS)
@pytest.mark.parametrize("prec", ["f", "d"])
def test_c2c(torch_gpu, dims, vecs, size, prec):
    ct = np.complex64 if prec == "f" else np.complex128
    rng = np.random.default_rng(size)
    n_in = 1 + sum((a[0] - 1) * a[1] for a in dims + vecs)
    x = (rng.standard_normal(n_in) + 1j * rng.standard_normal(n_in)).astype(ct)
    out = np.full(size, 7.5 - 2.5j, ct)
    ref = out.astype(np.complex128)
    O.c2c_strided(x.astype(np.complex128), ref, dims, vecs, -1)
    p = fftz.Plan(dims, vecs, prec, 0, inp=x, out=out)
    assert p.execute() == 0
    p.destroy()
    assert O.rel_l2(out, ref) <= tol(int(np.prod([d[0] for d in dims])), prec)
    gaps = np.ones(size, bool)
    idx = np.zeros(1, int)
    for n, _, s in dims + vecs:
        idx = (idx[:, None] + np.arange(n) * s).reshape(-1)
    gaps[idx] = False
    assert np.all(out[gaps] == ct(7.5 - 2.5j)) and gaps.any() == ((dims, vecs, size) in GAPS)


def test_real_dense(torch_gpu):
    n, b = 30, 4
    x = np.random.default_rng(1).standard_normal((b, n))
    y = np.full((b, n // 2 + 1), np.nan, np.complex128)
    back = np.full((b, n), np.nan)
    p = fftz.Plan([(n, 1, 1)], [(b, n, n // 2 + 1)], "d", 0, fft_type=1, inp=x, out=y)
    q = fftz.Plan([(n, 1, 1)], [(b, n // 2 + 1, n)], "d", 1, fft_type=1, inp=y, out=back)
    assert p.execute() == 0 and q.execute() == 0
    assert O.rel_l2(y, np.fft.rfft(x)) <= tol(n, "d")
    assert np.max(np.abs(back / n - x)) <= 1e-13
