"""Rounding of a row in FP32 (GPU).  The operator has one image per row at most, so
on a reduced space y_r = sqrt(N_r / G) (a sqrt(G / N_s) x_s) is rounded at most where
the scaled x is stored, where it is weighed and where y is: 3 x 2^-24 of it, and with
no sign of its own, so that the mean over M rows stays below 6 sigma, 6 x 3 /
sqrt(3 M) x 2^-24.  A factor common to all rows and rounded to FP32, as sqrt(N_r) and
1 / sqrt(N_s), would be off in every row alike, by up to 0.76 x 2^-24 on 18 sites and
0.61 on 24.  The FP64 product's own error is 1e-9 of that."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Lx,Ly,lookup", [(3, 6, "auto"), (24, 1, "auto"), (5, 6, "auto"), (3, 6, "bitmap"), (24, 1, "bitmap")])
def test_single_images(ed, Lx, Ly, lookup):
    n = Lx * Ly
    hs, s = ed.spin_half_system(n)
    space = ed.represent(ed.HilbertSpaceSector(hs, 0 if n < 28 else n - 12))
    irrep = ed.TranslationIrrep(n, 0) if Ly == 1 else ed.TranslationIrrep((Lx, Ly), (0, 0))
    opr = ed.represent(ed.symmetry_reduce(space, irrep), ed.PureOperator(3, 1, 2, 0.6875))
    if lookup != "auto":
        opr.set_strategy("terms", lookup)
    x = 1 + 0.5 * torch.rand(opr.dimension, device="cuda", generator=torch.Generator(device="cuda").manual_seed(n))
    y, z, wide = torch.empty_like(x), torch.empty(opr.dimension, dtype=torch.float64, device="cuda"), x.double()
    ed.mul_(y, opr, x)
    ed.mul_(z, opr, wide)
    rows = z > 0
    error = ((y.double() - z)[rows] / z[rows]) * 2.0**24
    M = int(rows.sum())
    assert M > opr.dimension // 8 and bool((y[~rows] == 0).all())
    assert float(error.abs().max()) <= 3 * (1 + 1e-6)
    assert abs(float(error.mean())) <= 6 * 3 / math.sqrt(3 * M)
