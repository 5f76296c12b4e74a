"""The term pass by rank (sectors of one popcount without a group) against the
general kernels (edhip_term_expect_noalloc, which never takes it), term by term:
word lengths around the split of the rank tables, both table sizes, all vector
types, terms alone and in pairs, diagonal terms of one to three sites on either
side of the split.  Both add the same products in double in other orders:
sums of D values of random sign, rounded at most once per addition, so the
difference stays below eps * sqrt(D) * sum |p| ~ 1e-12 of the largest form."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _operator(ed, n, rng):
    terms = []
    for _ in range(10):  # pairs that follow each other, and hops one way
        i, j = (1 << int(k) for k in rng.choice(n, 2, replace=False))
        terms.append(ed.PureOperator(i | j, i, j, 1.0))
        if rng.random() < 0.6:
            terms.append(ed.PureOperator(i | j, j, i, 1.0))
    for _ in range(12):
        sites = [int(k) for k in rng.choice(n, int(rng.integers(1, 3)), replace=False)]
        mask = sum(1 << k for k in sites)
        match = sum(1 << k for k in sites if rng.random() < 0.5)
        terms.append(ed.PureOperator(mask, match, match, 1.0))
    lower = sorted(rng.choice(11, 3, replace=False))  # three sites below the split
    terms.append(ed.PureOperator(sum(1 << int(k) for k in lower), 1 << int(lower[0]), 1 << int(lower[0]), 1.0))
    return ed.SumOperator(terms)


@pytest.mark.parametrize("n,up", [(12, 5), (13, 6), (16, 8), (18, 4), (24, 5), (25, 20), (26, 6)])
@pytest.mark.parametrize("wide", [False, True])
def test_ranked_term_pass(ed, n, up, wide):
    import torch

    from edhip import _lib

    hs, _ = ed.spin_half_system(n)
    rng = np.random.default_rng(n)
    op = _operator(ed, n, rng)
    if wide:  # two lower bits beside an upper one (where there is one): the general kernels
        op = op + ed.PureOperator(3 | 1 << (n - 1), 1, 1, 1.0)
    opr = ed.represent(ed.represent(ed.HilbertSpaceSector(hs, n - 2 * up)), op)
    L = _lib.lib()
    g = torch.Generator(device="cuda").manual_seed(n)
    for prec, dt in ((_lib.F64, torch.float64), (_lib.C128, torch.complex128), (_lib.F32, torch.float32),
                     (_lib.C64, torch.complex64)):
        phi = torch.randn(opr.dimension, dtype=dt, device="cuda", generator=g)
        psi = torch.randn(opr.dimension, dtype=dt, device="cuda", generator=g)
        torch.cuda.synchronize()
        a, b = np.zeros(2 * opr._n_terms), np.full(2 * opr._n_terms, np.nan)
        for fn, out in ((L.edhip_term_expect, a), (L.edhip_term_expect_noalloc, b)):
            opr.ctx.check(fn(opr._handle, prec, ctypes.c_void_p(phi.data_ptr()), ctypes.c_void_p(psi.data_ptr()),
                             out.ctypes.data_as(ctypes.POINTER(ctypes.c_double))))
        assert np.abs(b).max() > 0 and np.abs(a - b).max() <= 1e-12 * np.abs(b).max(), dt
