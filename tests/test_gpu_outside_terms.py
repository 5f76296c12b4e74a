"""Operators with terms on bits past the words of the space: such a term leads no
basis word to another, and the products and the term pass drop it, on every path
that finds images by their position (GPU, against the oracle).  At most 200 images
of weight below 2 per row: 1e-13 (2e-6) of the norm; the forms are sums of D
products: 1e-12 of the largest."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _operator(ed, hs, n, bonds):
    """Exchange on bonds, and terms with bits n and beyond in row, column, mask or all."""
    P = ed.PureOperator
    H = sum((ed.heisenberg_bond(hs, i, j, 1.0, 1.1) for i, j in bonds), ed.NullOperator())
    extra = []
    for top in (1 << n, 1 << (n + 4), 1 << 35, 1 << 62):
        extra += [P(1 | top, 1, top, 0.8), P(1 | top, top, 1, 0.8), P(2 | top, 0, 2 | top, 0.7), P(top, 0, top, 0.9),
                  P(top, top, 0, 0.9), P(7 | top, 1 | top, 2 | top, 0.4)]
    extra.append(P(1 << (n - 1) | 1 << (n - 2), 1 << (n - 1), 1 << (n - 2), 0.6))  # one way
    return ed.SumOperator(list(H.terms) + extra)


def _spaces(ed, oracle, n, up, irrep=None):
    hs, _ = ed.spin_half_system(n)
    space, basis = ed.represent(ed.HilbertSpaceSector(hs, n - 2 * up)), oracle.sector_basis(n, n - 2 * up)
    if irrep is None:
        return hs, space, basis
    pairs = list(irrep.symops_and_amplitudes())
    red = oracle.symmetry_reduce(basis, n, np.stack([ed.bit_permutation(hs, p) for p, _ in pairs]), [a for _, a in pairs])
    return hs, ed.symmetry_reduce(space, irrep), red


def _bonds(ed, n, shape):
    if shape is None or shape[1] == 1:
        return ed.chain_bonds(n)
    near, far = ed.square_bonds(*shape)
    return near + far


# rank tables of both sizes, the spread without a group, translations in 32- and
# 64-bit words, chains, point operations
CASES = [(16, 8, None, None), (24, 4, None, None), (25, 3, None, None), (26, 3, None, None), (28, 3, None, None), (27, 7, None, None),
         (16, 8, (4, 4), (1, 2)), (24, 5, (4, 6), (0, 0)), (25, 4, (5, 5), (1, 0)), (36, 3, (6, 6), (2, 0)),
         (13, 6, (13, 1), 3), (33, 3, (33, 1), 0), (25, 4, (5, 5), "A1"), (36, 4, (6, 6), "B1")]


@pytest.mark.parametrize("n,up,shape,k", CASES)
def test_products(ed, oracle, n, up, shape, k):
    import torch

    irrep = None
    if isinstance(k, str):
        irrep = ed.SquareSpaceIrrep(shape[0], (0, 0), k)
    elif shape is not None:
        irrep = ed.TranslationIrrep(n, k) if shape[1] == 1 else ed.TranslationIrrep(shape, k)
    hs, space, ospace = _spaces(ed, oracle, n, up, irrep)
    H = _operator(ed, hs, n, _bonds(ed, n, shape))
    opr, o = ed.represent(space, H), oracle.Opr(ospace, ed.terms_arrays(H))
    rng = np.random.default_rng(n)
    x = rng.standard_normal(opr.dimension) + (1j * rng.standard_normal(opr.dimension) if opr.is_complex else 0.0)
    for transpose in (False, True):
        ref = o.apply(np.zeros(opr.dimension, complex), x, transpose)
        for dt, tol in ((torch.complex128, 1e-13), (torch.complex64, 2e-6)):
            v = torch.tensor(x).to(dt if opr.is_complex else {torch.complex128: torch.float64}.get(dt, torch.float32)).cuda()
            y = torch.empty_like(v)
            ed.mul_(y, v, opr) if transpose else ed.mul_(y, opr, v)
            assert np.linalg.norm(y.cpu().numpy() - ref) <= tol * np.linalg.norm(ref), (dt, transpose)
    if irrep is not None:
        opr.set_strategy("assembled")
        ref = o.matvec(x)
        assert np.linalg.norm(opr @ x - ref) <= 1e-13 * np.linalg.norm(ref)
        opr.set_strategy()


def _forms(oracle, ospace, terms, phi, psi):
    mask, row, col, _ = terms
    one = np.ones(1)
    return np.array([np.vdot(phi, oracle.Opr(ospace, (mask[t:t + 1], row[t:t + 1], col[t:t + 1], one)).matvec(psi))
                     for t in range(len(mask))])


@pytest.mark.parametrize("n,up,shape,k", [CASES[i] for i in (0, 1, 3, 4, 6, 10)])
def test_term_pass(ed, oracle, n, up, shape, k):
    import torch

    irrep = None if shape is None else ed.TranslationIrrep(n, k) if shape[1] == 1 else ed.TranslationIrrep(shape, k)
    hs, space, ospace = _spaces(ed, oracle, n, up, irrep)
    H = _operator(ed, hs, n, _bonds(ed, n, shape)[:6])
    opr = ed.represent(space, H)
    rng = np.random.default_rng(n)
    phi, psi = (rng.standard_normal(opr.dimension) + 1j * rng.standard_normal(opr.dimension) for _ in range(2))
    ref = _forms(oracle, ospace, ed.terms_arrays(H), phi, psi)
    got = ed.term_expectations(opr, torch.tensor(phi).cuda(), torch.tensor(psi).cuda())
    assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("n,up", [(16, 8), (24, 4), (26, 3)])
@pytest.mark.parametrize("top", [0, 4, 35, 40, 62])
def test_diagonal_terms_past_the_words(ed, oracle, n, up, top):
    """Diagonal terms that test such a bit beside the forms by rank: no row has it set."""
    import torch

    hs, space, basis = _spaces(ed, oracle, n, up)
    P, bit, last = ed.PureOperator, 1 << (top if top > n else n + top), 1 << (n - 1)
    H = sum((ed.heisenberg_bond(hs, i, j) for i, j in ed.chain_bonds(n)[:4]), ed.NullOperator())
    H = ed.SumOperator(list(H.terms) + [P(1 | bit, 1 | bit, 1 | bit, 1.0), P(bit, bit, bit, 1.0), P(last | bit, bit, bit, 1.0),
                                        P(last | bit, last, last, 1.0), P(bit, 0, 0, 1.0), P(1 | bit, 0, 0, 1.0)])
    opr = ed.represent(space, H)
    rng = np.random.default_rng(n)
    phi, psi = rng.standard_normal((2, opr.dimension))
    ref = _forms(oracle, basis, ed.terms_arrays(H), phi, psi)
    got = ed.term_expectations(opr, torch.tensor(phi).cuda(), torch.tensor(psi).cuda())
    assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()
    y = opr @ psi
    ref = oracle.Opr(basis, ed.terms_arrays(H)).matvec(psi)
    assert np.linalg.norm(y - ref) <= 1e-13 * np.linalg.norm(ref)
