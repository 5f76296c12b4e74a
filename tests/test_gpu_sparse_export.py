"""The sparse matrix as it comes to the host through the staging buffers, against
the plain export of the same matrix (exactly), in both index sizes, real and
complex, over several staging parts and a last partial one (GPU)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Lx,Ly,k", [(4, 4, (1, 0)), (4, 5, (1, 2)), (4, 6, (2, 0)), (5, 5, (1, 1))])
def test_staged_export(ed, Lx, Ly, k):
    from edhip import _lib

    hs, _ = ed.spin_half_system(Lx * Ly)
    near, far = ed.square_bonds(Lx, Ly)
    H = sum((ed.heisenberg_bond(hs, i, j) for i, j in near), ed.NullOperator())
    H = ed.simplify(H + sum((ed.heisenberg_bond(hs, i, j, 0.3) for i, j in far), ed.NullOperator()))
    space = ed.represent(ed.HilbertSpaceSector(hs, Lx * Ly % 2))
    opr = ed.represent(ed.symmetry_reduce(space, ed.TranslationIrrep((Lx, Ly), k)), H)
    A = opr.sparse()
    n, nnz = opr.dimension, A.nnz
    assert A.indices.dtype == np.int32 and A.indptr.dtype == np.int32 and A.has_sorted_indices
    colptr, rowval = np.empty(n + 1, np.int64), np.empty(nnz, np.int64)
    re, im = np.empty(nnz), np.empty(nnz)
    L, i64, dbl = _lib.lib(), ctypes.c_int64, ctypes.c_double
    opr.ctx.check(L.edhip_sparse_export(opr._handle, _lib.ptr(colptr, i64), _lib.ptr(rowval, i64), _lib.ptr(re, dbl),
                                        _lib.ptr(im, dbl)))
    assert np.array_equal(A.indptr, colptr) and np.array_equal(A.indices, rowval)
    assert np.array_equal(A.data.real, re) and (not opr.is_complex or np.array_equal(A.data.imag, im))
    wide_ptr, wide_row, data = np.empty_like(colptr), np.empty_like(rowval), np.empty_like(A.data)
    opr.ctx.check(L.edhip_sparse_export_csc(opr._handle, 8, wide_ptr.ctypes.data_as(ctypes.c_void_p),
                                            wide_row.ctypes.data_as(ctypes.c_void_p), _lib.ptr(data, dbl)))
    assert np.array_equal(wide_ptr, colptr) and np.array_equal(wide_row, rowval) and np.array_equal(data, A.data)
    assert L.edhip_sparse_export_csc(opr._handle, 2, wide_ptr.ctypes.data_as(ctypes.c_void_p),
                                     wide_row.ctypes.data_as(ctypes.c_void_p), _lib.ptr(data, dbl)) != 0


@pytest.mark.parametrize("ranges", [1, 2, 5])
@pytest.mark.parametrize("k", [(0, 0), (1, 0)])
def test_columns_by_waves_and_by_lanes(ed, ranges, k):
    """Columns of at most 256 possible entries are merged by a wave, longer ones by
    a lane: both against the dense matrix, which sums term by term (at most 300
    terms below 1 per element: 1e-13), with entries that cancel (chopped) and
    rows of the transpose."""
    L = 4
    hs, _ = ed.spin_half_system(L * L)
    at = lambda x, y: (x % L) + L * (y % L)  # noqa: E731
    H = ed.NullOperator()
    for q, (dx, dy) in enumerate([(1, 0), (0, 1), (1, 1), (1, -1), (2, 0), (0, 2), (2, 1), (1, 2), (2, 2), (2, -1)][: 2 * ranges]):
        for x in range(L):
            for y in range(L):
                H = H + ed.heisenberg_bond(hs, at(x, y), at(x + dx, y + dy), 1.0 / (q + 1), 0.8)
    space = ed.symmetry_reduce(ed.represent(ed.HilbertSpaceSector(hs, 10)), ed.TranslationIrrep((L, L), k))
    opr = ed.represent(space, ed.simplify(H))
    A, M = opr.sparse(), opr.Matrix()
    assert A.has_sorted_indices and np.abs(A.toarray() - M).max() <= 1e-13 and abs(A.data).min() > 1e-9
    for i in (0, opr.dimension - 1):
        assert np.abs(opr.get_row(i).toarray()[0] - M[i]).max() <= 1e-13
        assert np.abs(opr.get_column(i).toarray()[:, 0] - M[:, i]).max() <= 1e-13
