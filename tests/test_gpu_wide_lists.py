"""Basis lists whose words have bits past those of the Hilbert space, and operators
that test them, against sums term by term (GPU): exchange bonds and fields, matched
by parity, and hops one way, matched by mask.  At most 40 terms below 2 per row:
1e-13."""
import numpy as np
import pytest

from conftest import dense_from_terms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,wide", [(4, 13), (10, 40), (12, 12), (12, 25), (30, 63)])
def test_products(ed, n, wide):
    rng = np.random.default_rng(wide)
    hs, _ = ed.spin_half_system(n)
    P = ed.PureOperator
    sites = rng.choice(wide, 4, replace=False)
    terms = []
    for i, j in [(0, wide - 1), (n - 1, wide - 2), *((int(a), int(b)) for a, b in zip(sites, sites[1:]))]:
        a, b = 1 << i, 1 << j
        for r, c, v in ((0, 0, 0.5), (a, a, -0.5), (b, b, -0.5), (a | b, a | b, 0.5), (a, b, 1.0), (b, a, 1.0)):
            terms.append(P(a | b, r, c, v))
    top = 1 << (wide - 1)
    terms += [P(top, 0, 0, 0.3), P(top, top, top, -0.3), P(top | 2, top, 2, 0.7), P(top, top, 0, 0.2), P(top, 0, top, 0.2)]
    words = {0, top, (1 << wide) - 1} | {int(w) for w in rng.integers(0, 1 << wide, 40, dtype=np.uint64)}
    for t in terms:  # images within the list
        words |= {(w & ~t.bitmask) | t.bitcol for w in list(words)[:60] if w & t.bitmask == t.bitrow}
    words = np.array(sorted(words), np.uint64)
    opr = ed.represent(ed.represent(hs, words), ed.SumOperator(terms))
    M = dense_from_terms(wide, words, ed.terms_arrays(ed.SumOperator(terms)))
    x = rng.standard_normal(words.size)
    assert np.abs(opr @ x - M.real @ x).max() <= 1e-13
    assert np.abs(x @ opr - x @ M.real).max() <= 1e-13
    assert np.abs(opr.Matrix() - M).max() <= 1e-13
