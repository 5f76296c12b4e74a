"""The sparse export over more blocks than one row of its grid holds (2^22, 16.8M
columns with a wave each): the matrix applied on the host against the product, in
small whole numbers, which both add exactly (GPU)."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_many_columns(ed):
    n, up = 27, 13
    hs, _ = ed.spin_half_system(n)
    P = ed.PureOperator
    H = ed.SumOperator([P(3, 1, 2, 3.0), P(1 << 26 | 4, 1 << 26, 4, 2.0), P(1 << 20, 1 << 20, 1 << 20, 5.0)])
    opr = ed.represent(ed.represent(ed.HilbertSpaceSector(hs, n - 2 * up)), H)
    A = opr.sparse()
    D = math.comb(n, up)
    assert opr.dimension == D > 1 << 24
    assert A.nnz == 2 * math.comb(n - 2, up - 1) + math.comb(n - 1, up - 1)
    x = np.arange(D, dtype=np.float64) % 97 + 1.0
    assert np.array_equal(A @ x, opr @ x)
