"""Products through parity entries, single terms and both, with one or several
lanes per row, against the oracle (GPU).  Tolerance: one rounding per image and
one per partial sum, at most a few hundred of them: 1e-13 relative in FP64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


def _bonds(n, count):
    pairs = [(i, j) for i in range(n) for j in range(i + 1, n)]
    return [pairs[k % len(pairs)] for k in range(count)]


# 1, 63, 64, 65 and 120 parity entries (segments of 64); asymmetric flips
# (S+S- alone) and transverse fields beside them; a full space, so that the
# fields stay inside; 2^10 to 2^13 rows (several lanes per row)
@pytest.mark.parametrize("n,count", [(10, 1), (12, 63), (12, 64), (13, 65), (16, 120)])
@pytest.mark.parametrize("extra", ["none", "hop", "field"])
def test_products_vs_oracle(ed, oracle, n, count, extra):
    rng = np.random.default_rng(100 * n + count)
    hs, s = ed.spin_half_system(n)
    ops = [ed.heisenberg_bond(hs, i, j, float(J)) for (i, j), J in zip(_bonds(n, count), rng.uniform(0.5, 1.5, count))]
    if extra == "hop":
        ops += [float(rng.uniform(0.2, 0.8)) * s(i, "+") * s((i + 2) % n, "-") for i in range(0, n, 3)]
    if extra == "field":
        ops += [0.3 * s(i, "x") for i in range(n)]
    H = ed.simplify(sum(ops, ed.NullOperator()))
    if extra == "field" and n > 13:
        pytest.skip("the full space of 16 sites repeats the smaller cases")
    space = ed.represent(hs if extra == "field" else ed.HilbertSpaceSector(hs, n % 2))
    opr = ed.represent(space, H)
    o = oracle.Opr(space.basis_list, ed.terms_arrays(H))
    x = rng.standard_normal(opr.dimension)
    assert rel(opr @ x, o.matvec(x).real) < 1e-13
    # the column form is the transpose of the row form
    z = rng.standard_normal(opr.dimension)
    assert abs(np.dot(z @ opr, x) - np.dot(z, opr @ x)) < 1e-12 * np.linalg.norm(z) * np.linalg.norm(opr @ x)
