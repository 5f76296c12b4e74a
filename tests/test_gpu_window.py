"""Products on translation-reduced tori and chains through the kernels of their
shape (window canonicaliser, 32- and 64-bit words) against the general kernels
with the blocked rank index (GPU).  Both sum the same few hundred images per
row in double (single) precision: 1e-13 (2e-6) relative."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.float64: 1e-13, torch.complex128: 1e-13, torch.float32: 2e-6, torch.complex64: 2e-6}


def _operator(ed, hs, s, Lx, Ly, kind):
    """Translation-invariant couplings: Heisenberg bonds, and beside them a
    complex hop (asymmetric amplitudes: matched term by term)."""
    at = lambda x, y: (x % Lx) + Lx * (y % Ly)  # noqa: E731
    steps = [(1, 0), (2, 0)] if Ly == 1 else [(1, 0), (0, 1), (1, 1)]
    ops = []
    for y in range(Ly):
        for x in range(Lx):
            for k, (a, b) in enumerate(steps):
                ops.append(ed.heisenberg_bond(hs, at(x, y), at(x + a, y + b), 1.0 - 0.4 * k, 1.1))
            if kind == "hop":
                i, j = at(x, y), at(x + 2, y + (Ly > 1))
                ops += [(0.3 + 0.2j) * s(i, "+") * s(j, "-"), (0.3 - 0.2j) * s(j, "+") * s(i, "-")]
    return ed.simplify(sum(ops, ed.NullOperator()))


# shapes on both sides of 4 windows, odd sides, rows of 7 and 8 bits; chains
# around multiples of 6 (whole and partial last windows) and past 32 bits
SHAPES = [(3, 6, 0, 0), (3, 7, 1, 2), (4, 5, 2, 0), (4, 6, 1, 3), (5, 4, 0, 2), (5, 5, 2, 1), (6, 3, 3, 0), (6, 4, 1, 1),
          (7, 3, 0, 0), (7, 3, 3, 1), (8, 3, 4, 0), (17, 1, 5, 0), (18, 1, 9, 0), (19, 1, 0, 0), (23, 1, 2, 0), (24, 1, 12, 0)]


@pytest.mark.parametrize("Lx,Ly,kx,ky", SHAPES)
@pytest.mark.parametrize("kind", ["heisenberg", "hop"])
def test_shape_kernel_vs_general(ed, Lx, Ly, kx, ky, kind):
    n = Lx * Ly
    hs, s = ed.spin_half_system(n)
    H = _operator(ed, hs, s, Lx, Ly, kind)
    irrep = ed.TranslationIrrep(n, kx) if Ly == 1 else ed.TranslationIrrep((Lx, Ly), (kx, ky))
    opr = ed.represent(ed.symmetry_reduce(ed.represent(ed.HilbertSpaceSector(hs, n % 2)), irrep), H)
    g = torch.Generator(device="cuda").manual_seed(n)
    for dt in [torch.complex128, torch.complex64] if opr.is_complex else list(TOL):
        x = torch.randn(opr.dimension, dtype=dt, device="cuda", generator=g)
        for form in ("row", "column"):
            y, z = torch.empty_like(x), torch.empty_like(x)
            opr.set_strategy("terms", "xspread")
            ed.mul_(y, opr, x) if form == "row" else ed.mul_(y, x, opr)
            opr.set_strategy("terms", "bitmap")
            ed.mul_(z, opr, x) if form == "row" else ed.mul_(z, x, opr)
            assert torch.linalg.norm(y - z) <= TOL[dt] * torch.linalg.norm(z), (dt, form)


@pytest.mark.parametrize("n", [33, 36])
def test_long_chain_few_flips(ed, n):
    """Chains past 32 sites (64-bit words): three up spins."""
    hs, s = ed.spin_half_system(n)
    H = _operator(ed, hs, s, n, 1, "heisenberg")
    hsr = ed.represent(ed.HilbertSpaceSector(hs, n - 6))
    for k in (0, 5):
        opr = ed.represent(ed.symmetry_reduce(hsr, ed.TranslationIrrep(n, k)), H)
        x = torch.randn(opr.dimension, dtype=torch.complex128, device="cuda")
        y, z = torch.empty_like(x), torch.empty_like(x)
        ed.mul_(y, opr, x)
        opr.set_strategy("terms", "search")
        ed.mul_(z, opr, x)
        assert torch.linalg.norm(y - z) <= 1e-13 * torch.linalg.norm(z)
