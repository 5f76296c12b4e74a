"""Diagonal elements of operators whose amplitudes the rows do not share: a row's
element is the sum of the terms that match it, whatever the others weigh, against
numpy sums rounded once (math.fsum over the matching terms).  An element may be
off by half a unit (1.2e-16 of it) and by what the carried errors round (1e-16)."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BIG = [1e3, 1e6, 1e8, 1e12, math.inf]


def _matching_sums(words, operator):
    parts = [[] for _ in words]
    for t in operator.terms:
        m, r, a = t.bitmask, t.bitrow, float(np.real(t.amplitude))
        assert r == t.bitcol
        for k, w in enumerate(words):
            if (w & m) == r:
                parts[k].append(a)
    return np.array([math.fsum(p) if all(map(math.isfinite, p)) else sum(p) for p in parts])


@pytest.mark.parametrize("big", BIG)
@pytest.mark.parametrize("kind", ["penalty", "projector", "identity"])
@pytest.mark.parametrize("reduced", [False, True])
def test_elements_of_untouched_rows(ed, big, kind, reduced):
    import torch

    n = 12
    hs, s = ed.spin_half_system(n)
    H = sum((0.37 * s(i, "z") * s((i + 1) % n, "z") for i in range(n)), ed.NullOperator())
    P = ed.PureOperator
    if kind == "penalty":  # on parallel pairs two sites apart
        for i in range(n):
            m = 1 << i | 1 << (i + 2) % n
            H = H + P(m, 0, 0, big) + P(m, m, m, big)
    else:  # on one site (every site where the space is reduced), and an identity that cancels it
        for i in range(n) if reduced else [3]:
            H = H + P(1 << i, 1 << i, 1 << i, -big)
        if kind == "identity":
            H = H + P(0, 0, 0, big)
    H = ed.SumOperator(list(H.terms))
    space = ed.represent(ed.HilbertSpaceSector(hs, 0))
    if reduced:
        space = ed.symmetry_reduce(space, ed.TranslationIrrep(n, 0))
    opr = ed.represent(space, H)
    x = torch.ones(opr.dimension, dtype=torch.float64, device="cuda")
    y = torch.empty_like(x)
    ed.mul_(y, opr, x)
    ref = _matching_sums([int(w) for w in space.basis_list], H)
    got, fin = y.cpu().numpy(), np.isfinite(ref)
    assert np.array_equal(np.isfinite(got), fin) and np.array_equal(got[~fin], ref[~fin], equal_nan=True)
    assert (np.abs(got[fin] - ref[fin]) <= 1.2e-16 * np.abs(ref[fin]) + 1e-16).all()
