"""The kernels of a new sector against plain restatements in numpy: the reduction by
windows (representatives exactly) and the diagonal elements by parities (sums of
at most 160 values below 1: 1e-13 of the largest)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(3, 6, 0, 0), (3, 6, 1, 3), (4, 4, 2, 1), (4, 5, 2, 0), (5, 4, 1, 2), (6, 3, 3, 0), (7, 3, 0, 1), (8, 3, 4, 0),
          (12, 1, 6, 0), (13, 1, 5, 0), (18, 1, 9, 0), (20, 1, 0, 0), (33, 1, 11, 0)]


def _rotations(w, n, perms):
    out = np.empty((len(perms), len(w)), np.uint64)
    for g, p in enumerate(perms):
        v = np.zeros_like(w)
        for i, j in enumerate(p):
            v |= ((w >> np.uint64(i)) & np.uint64(1)) << np.uint64(j)
        out[g] = v
    return out


@pytest.mark.parametrize("Lx,Ly,kx,ky", SHAPES)
def test_reduction_and_diagonal(ed, Lx, Ly, kx, ky):
    import torch

    n = Lx * Ly
    up = 3 if n > 24 else n // 2
    hs, s = ed.spin_half_system(n)
    hsr = ed.represent(ed.HilbertSpaceSector(hs, n - 2 * up))
    irrep = ed.TranslationIrrep(n, kx) if Ly == 1 else ed.TranslationIrrep((Lx, Ly), (kx, ky))
    pairs = list(irrep.symops_and_amplitudes())
    red = ed.symmetry_reduce(hsr, irrep)
    words = np.array(hsr.basis_list, dtype=np.uint64)
    perms = [ed.bit_permutation(hs, p) for p, _ in pairs]
    chi = np.array([complex(a) for _, a in pairs])
    img = _rotations(words, n, perms)
    fixed = img == words
    keep = (img >= words).all(axis=0) & ~(fixed & (np.abs(chi - 1) > 1e-8)[:, None]).any(axis=0)
    assert np.array_equal(np.array(red.basis_list, dtype=np.uint64), words[keep])
    # diagonal: pairs of two strengths, one-site fields, a three-site term (1: bit 0, -1: bit 1)
    reps = words[keep]
    z = [1.0 - 2.0 * ((reps >> np.uint64(i)) & np.uint64(1)).astype(float) for i in range(n)]
    H, ref = ed.NullOperator(), np.zeros(len(reps))
    for c, k in ((1.0, 1), (0.37, 2)):
        for i, j in sorted({tuple(sorted((int(p[0]), int(p[k])))) for p in perms}):
            H, ref = H + c * s(i, "z") * s(j, "z"), ref + c * z[i] * z[j]
    for i in range(n):
        H, ref = H + 0.25 * s(i, "z"), ref + 0.25 * z[i]
    for i, j, k in sorted({tuple(int(p[q]) for q in (0, 1, 2)) for p in perms}):
        H, ref = H + 0.2 * s(i, "z") * s(j, "z") * s(k, "z"), ref + 0.2 * z[i] * z[j] * z[k]
    opr = ed.represent(red, ed.simplify(H))
    dt = torch.complex128 if opr.is_complex else torch.float64
    x = torch.ones(opr.dimension, dtype=dt, device="cuda")
    y = torch.empty_like(x)
    ed.mul_(y, opr, x)
    assert np.abs(y.cpu().numpy() - ref).max() <= 1e-13 * max(1.0, np.abs(ref).max())
