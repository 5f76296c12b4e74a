"""Products on every torus shape compiled with a kernel of its own, and on chains
(longer ones, whose small sectors are too sparse for the spread, on the CPU alone),
against the oracle, with the kernel that ran named (GPU).  Shapes past 24 sites in
sectors of four up spins.  Rows sum a few hundred images: 1e-13 (2e-6) relative."""
import ctypes
import os
import re

import numpy as np
import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

SHAPE, POINT, RANK = 2, 3, 4
with open(os.path.join(ROOT, "exactdiagonalization.jl_amd", "csrc", "window.hpp")) as f:
    SHAPES = [(int(a), int(b)) for a, b in re.findall(r"X\(kWin\w+, (\d+), (\d+)\)", f.read())]
CHAINS = [(n, 1) for n in (17, 24, 31, 32, 33, 36)]


def _path(opr, product=True):
    from edhip import _lib

    p, t = ctypes.c_int(), ctypes.c_int()
    opr.ctx.check(_lib.lib().edhip_debug_paths(opr._handle, ctypes.byref(p), ctypes.byref(t)))
    return p.value if product else t.value


def _operator(ed, hs, s, Lx, Ly, hop):
    at = lambda x, y: (x % Lx) + Lx * (y % Ly)  # noqa: E731
    steps = [(1, 0), (2, 0)] if Ly == 1 else [(1, 0), (0, 1), (1, 1)]
    H = ed.NullOperator()
    for y in range(Ly):
        for x in range(Lx):
            for k, (a, b) in enumerate(steps):
                H = H + ed.heisenberg_bond(hs, at(x, y), at(x + a, y + b), 1.0 - 0.4 * k, 1.1)
            if hop:  # matched term by term
                i, j = at(x, y), at(x + 2, y + (Ly > 1))
                H = H + (0.3 + 0.2j) * s(i, "+") * s(j, "-") + (0.3 - 0.2j) * s(j, "+") * s(i, "-")
    return ed.simplify(H)


def test_all_shapes_are_listed():
    assert len(SHAPES) == 21 and (7, 5) in SHAPES and (5, 7) in SHAPES


@pytest.mark.parametrize("Lx,Ly", SHAPES + CHAINS)
@pytest.mark.parametrize("complex_", [False, True])
def test_shape(ed, oracle, Lx, Ly, complex_):
    import torch

    n = Lx * Ly
    up = n // 2 if n <= 18 else 6 if n <= 24 else 4
    hs, s = ed.spin_half_system(n)
    k = (1 if complex_ else 0, Ly // 2 if complex_ else 0)
    irrep = ed.TranslationIrrep(n, k[0]) if Ly == 1 else ed.TranslationIrrep((Lx, Ly), k)
    space = ed.symmetry_reduce(ed.represent(ed.HilbertSpaceSector(hs, n - 2 * up)), irrep)
    pairs = list(irrep.symops_and_amplitudes())
    red = oracle.symmetry_reduce(oracle.sector_basis(n, n - 2 * up), n, np.stack([ed.bit_permutation(hs, p) for p, _ in pairs]),
                                 [a for _, a in pairs])
    assert np.array_equal(space.basis_list, red.basis_list)
    H = _operator(ed, hs, s, Lx, Ly, complex_)
    opr, o = ed.represent(space, H), oracle.Opr(red, ed.terms_arrays(H))
    assert opr.is_complex == complex_
    rng = np.random.default_rng(n)
    x = rng.standard_normal(opr.dimension) + (1j * rng.standard_normal(opr.dimension) if complex_ else 0.0)
    types = [(torch.complex128, 1e-13), (torch.complex64, 2e-6)]
    if not complex_:
        types += [(torch.float64, 1e-13), (torch.float32, 2e-6)]
    # (the kernels of a shape need words of 16 bits and more)
    path = SHAPE if int(space.basis_list.max()).bit_length() >= 16 else 1
    for transpose in (False, True):
        ref = o.apply(np.zeros(opr.dimension, complex), x, transpose)
        for dt, tol in types:
            v = torch.tensor(x).to(dt).cuda()
            y = torch.empty_like(v)
            ed.mul_(y, v, opr) if transpose else ed.mul_(y, opr, v)
            assert _path(opr) == path
            assert np.linalg.norm(y.cpu().numpy() - ref) <= tol * np.linalg.norm(ref), (dt, transpose)


def test_other_paths(ed):
    """The kernels by rank and of the point operations run where they are meant to."""
    for n, up, product in ((12, 6, RANK), (24, 4, RANK), (26, 3, RANK), (27, 7, SHAPE)):
        hs, _ = ed.spin_half_system(n)
        H = sum((ed.heisenberg_bond(hs, i, j) for i, j in ed.chain_bonds(n)), ed.NullOperator())
        opr = ed.represent(ed.represent(ed.HilbertSpaceSector(hs, n - 2 * up)), ed.simplify(H))
        opr @ np.ones(opr.dimension)
        assert _path(opr) == product
        ones = np.ones(opr.dimension)
        import torch

        ed.term_expectations(opr, torch.tensor(ones).cuda(), torch.tensor(ones).cuda())
        assert _path(opr, product=False) == (RANK if n <= 26 else 1)
    for L, up in ((5, 6), (6, 5)):
        hs, _ = ed.spin_half_system(L * L)
        near, _ = ed.square_bonds(L, L)
        H = ed.simplify(sum((ed.heisenberg_bond(hs, i, j) for i, j in near), ed.NullOperator()))
        space = ed.symmetry_reduce(ed.represent(ed.HilbertSpaceSector(hs, L * L - 2 * up)), ed.SquareSpaceIrrep(L, (0, 0), "A1"))
        opr = ed.represent(space, H)
        opr @ np.ones(opr.dimension)
        assert _path(opr) == POINT
