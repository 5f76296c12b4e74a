"""Device memory of small objects (GPU): their tables share slabs, an object's own
part is its tables', and objects freed in any order leave the others' tables as
they are.  The limits are what a program paid with an allocation per table (17 and
18 of 4 kB)."""
import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _free():
    import torch

    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def _operator(ed, hs, space, q):
    return ed.represent(space, ed.simplify(sum((ed.heisenberg_bond(hs, i, (i + 1) % 8, 1.0 + q) for i in range(8)),
                                               ed.NullOperator())))


def test_small_operators(ed):
    hs, _ = ed.spin_half_system(8)
    space = ed.represent(ed.HilbertSpaceSector(hs, 0))
    x = np.random.default_rng(0).standard_normal(space.dimension)
    unit = _operator(ed, hs, space, 0) @ x
    before = _free()
    ops = [_operator(ed, hs, space, q) for q in range(400)]
    assert (before - _free()) / len(ops) < 68e3
    for q in range(0, 400, 3):  # some end, in an order of their own
        ops[(7 * q) % 400] = None
    gc.collect()
    more = [_operator(ed, hs, space, q) for q in range(30)]
    for q, o in list(enumerate(ops)) + list(enumerate(more)):
        if o is not None and q % 10 == 0:
            assert np.linalg.norm(o @ x - (1.0 + q) * unit) <= 1e-13 * (1 + q) * np.linalg.norm(unit)


def test_small_reductions(ed):
    hs, _ = ed.spin_half_system(8)
    space = ed.represent(ed.HilbertSpaceSector(hs, 0))
    ed.symmetry_reduce(space, ed.TranslationIrrep(8, 0))
    before = _free()
    red = [ed.symmetry_reduce(space, ed.TranslationIrrep(8, q % 8)) for q in range(200)]
    assert (before - _free()) / len(red) < 73e3
