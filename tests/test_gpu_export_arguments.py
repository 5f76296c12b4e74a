"""The sparse export for the host refuses null outputs before anything is copied (GPU);
an empty matrix needs no room for its entries."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_null_outputs(ed):
    from edhip import _lib

    L, none = _lib.lib(), ctypes.c_void_p()
    hs, _ = ed.spin_half_system(8)
    space = ed.represent(ed.HilbertSpaceSector(hs, 0))
    opr = ed.represent(space, ed.simplify(sum((ed.heisenberg_bond(hs, i, (i + 1) % 8) for i in range(8)), ed.NullOperator())))
    A = opr.sparse()
    colptr, rowval, values = np.empty(A.shape[0] + 1, np.int32), np.empty(A.nnz, np.int32), np.empty(A.nnz)

    def export(o, p, r, v):
        at = [none if a is None else a.ctypes.data_as(ctypes.c_void_p) for a in (p, r)]
        return L.edhip_sparse_export_csc(o._handle, 4, *at, None if v is None else _lib.ptr(v, ctypes.c_double))

    for missing in range(3):
        out = [colptr, rowval, values]
        out[missing] = None
        assert export(opr, *out) == _lib.EDHIP_ERR_ARGUMENT
    assert export(opr, colptr, rowval, values) == 0
    assert np.array_equal(colptr, A.indptr) and np.array_equal(rowval, A.indices) and np.array_equal(values, A.data)
    empty = ed.represent(space, ed.NullOperator())
    assert empty.sparse().nnz == 0
    assert export(empty, colptr, None, None) == 0 and not colptr.any()
