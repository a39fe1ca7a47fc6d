"""What a plan reports about itself (no GPU): the kernel each launch gets -- form,
radix set, half exchange, stores past the L2 -- on both sides of the rules that
pick it, the LDS that is launched, stage strides, values per thread."""
import numpy as np
import pytest

import fftz

POW2, ALL, LIGHT, TO8 = 0, 1, 2, 3  # RadixSet, kernels.h


def only(dims, vecs, prec="f", direction=0, **k):
    ln = fftz.plan_json(dims, vecs, prec, direction, **k)["launches"]
    assert len(ln) == 1
    return ln[0]


@pytest.mark.parametrize("n,prec,form,rad", [
    (16, "f", "pass", POW2), (64, "f", "fixed", POW2), (8192, "f", "pass", POW2), (24, "f", "pass", LIGHT),
    (12, "f", "pass", LIGHT), (132, "f", "pass", LIGHT), (13, "f", "pass", ALL), (48, "f", "pass", ALL),
    (16, "d", "pass", POW2), (8, "d", "pass", TO8), (56, "d", "pass", TO8), (9, "d", "pass", LIGHT), (100, "d", "pass", LIGHT),
    (13, "d", "pass", ALL), (48, "d", "pass", ALL), (17, "f", "bluestein", None), (1009, "d", "bluestein", POW2)])
def test_form_and_radix_set(n, prec, form, rad):
    ln = only([(n, 1, 1)], [(4, n, n)], prec)
    assert ln["form"] == form and rad in (None, ln["rad"])


@pytest.mark.parametrize("half,prec,form,rad", [
    (6, "d", "real", TO8), (7, "d", "real", ALL), (36, "d", "real", ALL), (42, "d", "real", TO8), (49, "d", "real", ALL),
    (10, "f", "real", ALL), (11, "f", "real_wide", ALL), (143, "f", "real_wide", ALL), (16, "f", "real", POW2)])
@pytest.mark.parametrize("direction", [0, 1])
def test_real_form(half, prec, form, rad, direction):
    a, b = 2 * half, half + 1
    vec = (4, a, b) if direction == 0 else (4, b, a)
    ln = only([(a, 1, 1)], [vec], prec, direction, fft_type=1)
    assert ln["form"] == form and ln["rad"] == rad


def test_launched_lds_and_half_exchange():
    # 512-point columns of a volume: exchanges in halves, half of the tile is launched
    pj = fftz.plan_json([(512, 1, 1), (512, 512, 512), (512, 512 * 512, 512 * 512)], [(1, 1 << 27, 1 << 27)], "f")
    col = pj["launches"][1]
    assert col["split"] == 1 and 2 * col["lds_launched"] == col["C"] * col["LP"] * 8
    row = pj["launches"][0]
    assert row["split"] == 0 and row["lds_launched"] == row["C"] * row["LP"] * 8
    assert not row["nt"]  # read by the next launch


def test_stage_strides_and_batch_values_per_thread():
    ln = only([(1200, 1, 1)], [(4, 1200, 1200)])
    assert ln["ls"] == [int(np.prod(ln["radix"][:s])) for s in range(len(ln["radix"]))]
    pj = fftz.batch_plan_json([(16, 3, 0, 0), (1000, 2, 48, 48), (16384, 1, 2048, 2048)], "f")
    for c in pj["classes"]:
        most = max([-(-pj["sizes"][t[0]]["L"] // pj["sizes"][t[0]]["TL"]) for t in c["tiles"]], default=0)
        assert c["E"] == most


@pytest.mark.parametrize("n,batch,prec,nt", [
    (64, 4096, "f", 0), (1024, 4096, "f", 1), (1024, 8192, "f", 1), (100, 17, "f", 0), (1200, 3001, "f", 1),
    (1200, 3500, "f", 0), (1200, 17000, "f", 0), (1200, 18000, "f", 1), (1200, 4096, "d", 1), (1009, 1500, "d", 1),
    (1009, 4000, "d", 0), (1009, 11000, "d", 1)])
def test_stores_past_the_l2(n, batch, prec, nt):
    # rows of whole cache lines; not where a reader of the output loses more than the plan gains
    assert only([(n, 1, 1)], [(batch, n, n)], prec)["nt"] == nt


@pytest.mark.parametrize("n,batch,TL", [(4004, 261, 256), (4004, 256, 512), (4095, 1024, 256), (8190, 512, 512),
                                        (5005, 600, 512)])
def test_threads_of_complex128_rows(n, batch, TL):
    # 256 where the LDS holds two tiles and there are more lines than CUs
    assert only([(n, 1, 1)], [(batch, n, n)], "d")["TL"] == TL
