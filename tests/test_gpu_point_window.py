"""Products on the space groups of square tori through the window kernel of the
point operations against the general kernels with the sorted search (GPU),
for every little group it takes, unit and signed characters.  Both sum the same
few hundred images per row; the window kernel reads x / sqrt(N) rounded to the
vector's type: 1e-13 (2e-6) relative."""
import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.float64: 1e-13, torch.complex128: 1e-13, torch.float32: 2e-6, torch.complex64: 2e-6}

# (side, k, irrep, up spins away from half filling): C4v, C2v, Cs along an axis
# and along the diagonal (complex characters); the anti-diagonal mirror stays general
GROUPS = [(5, (0, 0), "A1", 0), (5, (0, 0), "B2", 0), (5, (0, 0), "A2", 2), (5, (0, 1), "A'", 4), (5, (1, 1), "A''", 4),
          (5, (1, 4), "A'", 4), (6, (0, 0), "A1", 10), (6, (3, 3), "B1", 10), (6, (3, 0), "B1", 10), (6, (2, 2), "A'", 12)]


@pytest.mark.parametrize("L,k,point,away", GROUPS)
@pytest.mark.parametrize("hop", [False, True])
def test_point_window_vs_general(ed, L, k, point, away, hop):
    n = L * L
    hs, s = ed.spin_half_system(n)
    near, far = ed.square_bonds(L, L)
    H = sum((ed.heisenberg_bond(hs, i, j, 1.0, 1.1) for i, j in near), ed.NullOperator())
    H = H + sum((ed.heisenberg_bond(hs, i, j, 0.4) for i, j in far), ed.NullOperator())
    if hop:  # four-site exchange round every plaquette: entries matched by mask
        at = lambda x, y: (x % L) + L * (y % L)  # noqa: E731
        for x in range(L):
            for y in range(L):
                a, b, c, d = at(x, y), at(x + 1, y), at(x + 1, y + 1), at(x, y + 1)
                H = H + 0.3 * (s(a, "+") * s(b, "-") * s(c, "+") * s(d, "-") + s(a, "-") * s(b, "+") * s(c, "-") * s(d, "+"))
    space = ed.represent(ed.HilbertSpaceSector(hs, n % 2 + 2 * away))
    opr = ed.represent(ed.symmetry_reduce(space, ed.SquareSpaceIrrep(L, k, point)), ed.simplify(H))
    g = torch.Generator(device="cuda").manual_seed(n)
    for dt in [torch.complex128, torch.complex64] if opr.is_complex else list(TOL):
        x = torch.randn(opr.dimension, dtype=dt, device="cuda", generator=g)
        for form in ("row", "column"):
            y, z = torch.empty_like(x), torch.empty_like(x)
            opr.set_strategy()
            ed.mul_(y, opr, x) if form == "row" else ed.mul_(y, x, opr)
            assert opr.last_strategy() == ("terms", "bitmap") or k == (1, 4)  # positions ranked
            opr.set_strategy("terms", "search")
            ed.mul_(z, opr, x) if form == "row" else ed.mul_(z, x, opr)
            assert torch.linalg.norm(y - z) <= TOL[dt] * torch.linalg.norm(z), (dt, form)
    opr.set_strategy()


@pytest.mark.parametrize("L,k,point,away", GROUPS)
def test_assembled_point_rows(ed, L, k, point, away):
    """The rows assembled through the window tables: the same products."""
    hs, _ = ed.spin_half_system(L * L)
    near, far = ed.square_bonds(L, L)
    H = sum((ed.heisenberg_bond(hs, i, j, 1.0, 1.1) for i, j in near), ed.NullOperator())
    H = H + sum((ed.heisenberg_bond(hs, i, j, 0.4) for i, j in far), ed.NullOperator())
    space = ed.represent(ed.HilbertSpaceSector(hs, L * L % 2 + 2 * away))
    opr = ed.represent(ed.symmetry_reduce(space, ed.SquareSpaceIrrep(L, k, point)), ed.simplify(H))
    g = torch.Generator(device="cuda").manual_seed(L)
    for dt in [torch.complex128, torch.complex64] if opr.is_complex else list(TOL):
        x = torch.randn(opr.dimension, dtype=dt, device="cuda", generator=g)
        y, z = torch.empty_like(x), torch.empty_like(x)
        opr.set_strategy("assembled")
        ed.mul_(y, opr, x)
        opr.set_strategy("terms", "search")
        ed.mul_(z, opr, x)
        assert torch.linalg.norm(y - z) <= TOL[dt] * torch.linalg.norm(z), dt
    opr.set_strategy()
