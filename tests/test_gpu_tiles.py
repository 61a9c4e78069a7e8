"""Row tiles built on the device (rows sorted, no repeats; the transpose's
tiles at every size, the matrix's own past a few thousand entries) against
the host build, which takes the same matrix with its rows' entries in another order:
the layouts are the same, so products are equal bit for bit; and against
numpy (1e-13 / 1e-5 of the largest entry)."""

import ctypes
import time

import numpy
import pytest
import scipy.sparse

from imate_amd import _lib

pytestmark = pytest.mark.gpu


def _banded(nrows, ncols, width, seed, dtype):
    """Dense-ish band (its 16-row tiles are well filled) with an empty row
    and one long row."""
    rng = numpy.random.default_rng(seed)
    M = scipy.sparse.lil_matrix((nrows, ncols), dtype=dtype)
    for r in range(nrows):
        c0 = min(max(0, r * ncols // nrows - width // 2), max(0, ncols - width))
        cols = numpy.arange(c0, min(ncols, c0 + width))
        cols = cols[rng.random(len(cols)) < 0.8]
        M[r, cols] = rng.standard_normal(len(cols)).astype(dtype)
    if nrows > 5:
        M[3, :] = 0
        M[5, :] = rng.standard_normal(ncols).astype(dtype)
    return M.tocsr()


def _shuffled(A, seed):
    rng = numpy.random.default_rng(seed)
    ix, dv = A.indices.copy(), A.data.copy()
    for r in range(A.shape[0]):
        p = rng.permutation(A.indptr[r + 1] - A.indptr[r]) + A.indptr[r]
        ix[A.indptr[r]:A.indptr[r + 1]] = A.indices[p]
        dv[A.indptr[r]:A.indptr[r + 1]] = A.data[p]
    return A.indptr, ix, dv


def _tiled(A, R):
    """Whether the tiled form is used: a quarter of its slab entries or more
    are non-zero (slab lists padded to eight for 16-row tiles). Without it
    products follow each row's entry order."""
    slabs = 0
    for t in range(0, A.shape[0], R):
        u = len(numpy.unique(A.indices[A.indptr[t]:
                                       A.indptr[min(t + R, A.shape[0])]]))
        slabs += -(-u // 8) * 8 if R == 16 else u
    return A.nnz >= 0.25 * slabs * R


def _handle(lib, shape, indptr, indices, data):
    ip = numpy.ascontiguousarray(indptr, dtype=numpy.int64)
    ix = numpy.ascontiguousarray(indices, dtype=numpy.int32)
    dv = numpy.ascontiguousarray(data)
    h = ctypes.c_void_p()
    _lib.check(lib.slq_op_create_csr(shape[0], shape[1], len(ix),
                                     _lib.ptr(ip), _lib.ptr(ix), _lib.ptr(dv),
                                     _lib.dtype_code(dv.dtype),
                                     ctypes.byref(h)), 'slq_op_create_csr')
    return h


def _spmm(lib, h, t, X, nrows, transpose=0):
    Y = numpy.empty((nrows, X.shape[1]), dtype=X.dtype)
    _lib.check(lib.slq_op_spmm(h, t, X.shape[1], transpose, _lib.ptr(X),
                               _lib.ptr(Y)), 'slq_op_spmm')
    return Y


@pytest.mark.parametrize('rows', ['16', '8'])
@pytest.mark.parametrize('dtype', [numpy.float64, numpy.float32])
@pytest.mark.parametrize('nrows,ncols,width', [
    (1, 1, 1), (7, 7, 7), (16, 16, 9), (17, 17, 5), (33, 90, 40),
    (200, 200, 64), (210, 300, 130)])
def test_device_tiles_equal_host_tiles(gpu_lib, monkeypatch, nrows, ncols,
                                       width, dtype, rows):
    monkeypatch.setenv('SLQ_TILE_ROWS', rows)
    A = _banded(nrows, ncols, width, nrows, dtype)
    h1 = _handle(gpu_lib, A.shape, A.indptr, A.indices, A.data)
    h2 = _handle(gpu_lib, A.shape, *_shuffled(A, 1))
    try:
        X = numpy.random.default_rng(2).standard_normal(
            (ncols, 64)).astype(dtype)
        Y1 = _spmm(gpu_lib, h1, 0.0, X, nrows)
        Y2 = _spmm(gpu_lib, h2, 0.0, X, nrows)
        if _tiled(A, int(rows)):
            assert numpy.array_equal(Y1, Y2)
        ref = A.astype(numpy.float64) @ X.astype(numpy.float64)
        tol = 1e-13 if dtype == numpy.float64 else 1e-5
        assert numpy.max(numpy.abs(Y1 - ref)) <= \
            tol * max(1.0, numpy.max(numpy.abs(ref)))
        Z = numpy.random.default_rng(3).standard_normal(
            (nrows, 64)).astype(dtype)
        Y1 = _spmm(gpu_lib, h1, 0.0, Z, ncols, 1)
        Y2 = _spmm(gpu_lib, h2, 0.0, Z, ncols, 1)
        if _tiled(A, int(rows)) and _tiled(A.T.tocsr(), int(rows)):
            assert numpy.array_equal(Y1, Y2)
        ref = A.T.astype(numpy.float64) @ Z.astype(numpy.float64)
        assert numpy.max(numpy.abs(Y1 - ref)) <= \
            tol * max(1.0, numpy.max(numpy.abs(ref)))
        # new values through the slot -> position map
        new = numpy.arange(1, A.nnz + 1).astype(dtype) / A.nnz
        _lib.check(gpu_lib.slq_op_set_values(h1, _lib.ptr(new)), 'values')
        B = scipy.sparse.csr_matrix((new, A.indices, A.indptr), shape=A.shape)
        ref = B.astype(numpy.float64) @ X.astype(numpy.float64)
        assert numpy.max(numpy.abs(_spmm(gpu_lib, h1, 0.0, X, nrows) - ref)) \
            <= tol * max(1.0, numpy.max(numpy.abs(ref)))
    finally:
        gpu_lib.slq_op_destroy(h1)
        gpu_lib.slq_op_destroy(h2)


@pytest.mark.parametrize('n', [5, 16, 17, 33, 50, 131])
def test_device_pair_tiles_equal_host(gpu_lib, n):
    A = _banded(n, n, 12, n, numpy.float64)
    B = _banded(n, n, 30, n + 1, numpy.float64)
    hs = []
    try:
        for a, b in ((A, B), (A, None)):
            ha = _handle(gpu_lib, A.shape, A.indptr, A.indices, A.data)
            hb = _handle(gpu_lib, B.shape, B.indptr, B.indices, B.data) \
                if b is not None else \
                _handle(gpu_lib, B.shape, *_shuffled(B, 3))
            hab = ctypes.c_void_p()
            _lib.check(gpu_lib.slq_op_create_affine(ha, hb, ctypes.byref(hab)),
                       'slq_op_create_affine')
            hs.append((hab, ha, hb))
        X = numpy.random.default_rng(n).standard_normal((n, 64))
        union = (abs(A) + abs(B)).tocsr()
        for t in (0.0, 0.75):
            Y = [_spmm(gpu_lib, h[0], t, X, n) for h in hs]
            if _tiled(A, 16) and _tiled(union, 16):
                assert numpy.array_equal(Y[0], Y[1])
            ref = A @ X + t * (B @ X)
            assert numpy.max(numpy.abs(Y[0] - ref)) <= \
                1e-13 * numpy.max(numpy.abs(ref))
    finally:
        for t in hs:
            for h in t:
                gpu_lib.slq_op_destroy(h)


def test_bad_column_is_named(gpu_lib):
    ip = numpy.array([0, 2, 3], dtype=numpy.int64)
    for bad in (2, -1):
        ix = numpy.array([0, 1, bad], dtype=numpy.int32)
        dv = numpy.ones(3)
        h = ctypes.c_void_p()
        code = gpu_lib.slq_op_create_csr(2, 2, 3, _lib.ptr(ip), _lib.ptr(ix),
                                         _lib.ptr(dv), _lib.SLQ_F64,
                                         ctypes.byref(h))
        assert code == _lib.SLQ_E_ARG
        assert 'column index %d out of range at 2' % bad in _lib.last_error()


# past a few thousand entries the columns are looked over on the device, with
# and without tiles to build, and the host names the one found
@pytest.mark.parametrize('rows', [None, '8', '0'])
@pytest.mark.parametrize('at', ['first', 'middle', 'last'])
def test_bad_column_of_a_larger_matrix(gpu_lib, monkeypatch, rows, at):
    if rows is None:
        monkeypatch.delenv('SLQ_TILE_ROWS', raising=False)
    else:
        monkeypatch.setenv('SLQ_TILE_ROWS', rows)
    n = 2000
    A = scipy.sparse.diags([4.0, 0.5, 0.5], [0, 1, -1], shape=(n, n),
                           format='csr')
    k = {'first': 0, 'middle': A.nnz // 2, 'last': A.nnz - 1}[at]
    ip = A.indptr.astype(numpy.int64)
    for bad in (n, -1, 2**31 - 1):
        ix = A.indices.astype(numpy.int32)
        ix[k] = bad
        h = ctypes.c_void_p()
        code = gpu_lib.slq_op_create_csr(n, n, A.nnz, _lib.ptr(ip),
                                         _lib.ptr(ix), _lib.ptr(A.data),
                                         _lib.SLQ_F64, ctypes.byref(h))
        assert code == _lib.SLQ_E_ARG
        assert 'column index %d out of range at %d' % (bad, k) in \
            _lib.last_error()


def _bordered(n, full, at, seed):
    """Tridiagonal with `full` full rows from row `at` on."""
    rng = numpy.random.default_rng(seed)
    A = scipy.sparse.diags([4.0 + rng.random(n), rng.random(n - 1),
                            rng.random(n - 1)], [0, 1, -1], format='lil')
    for r in range(at, at + full):
        A[r, :] = rng.standard_normal(n)
    return A.tocsr()


# a full row last in its tile and alone (no tiled form), a tile of full rows
# (tiled); the transpose and the union take the rows' lengths from the device
@pytest.mark.parametrize('n', [500, 2000])
@pytest.mark.parametrize('full,at', [(1, 15), (16, 16), (16, 24)])
def test_long_rows(gpu_lib, n, full, at):
    A = _bordered(n, full, at, n)
    B = _banded(n, n, 9, 3, numpy.float64)
    h1 = _handle(gpu_lib, A.shape, A.indptr, A.indices, A.data)
    h2 = _handle(gpu_lib, A.shape, *_shuffled(A, 1))
    hb = _handle(gpu_lib, B.shape, B.indptr, B.indices, B.data)
    hab = ctypes.c_void_p()
    _lib.check(gpu_lib.slq_op_create_affine(h1, hb, ctypes.byref(hab)),
               'slq_op_create_affine')
    try:
        X = numpy.random.default_rng(2).standard_normal((n, 64))
        for trans, M in ((0, A), (1, A.T.tocsr())):
            Y1 = _spmm(gpu_lib, h1, 0.0, X, n, trans)
            Y2 = _spmm(gpu_lib, h2, 0.0, X, n, trans)
            if _tiled(A, 16) and _tiled(M, 16):
                assert numpy.array_equal(Y1, Y2)
            ref = M @ X
            assert numpy.max(numpy.abs(Y1 - ref)) <= \
                1e-13 * numpy.max(numpy.abs(ref))
            ref = ref + 0.75 * ((B.T if trans else B) @ X)
            Y = _spmm(gpu_lib, hab, 0.75, X, n, trans)
            assert numpy.max(numpy.abs(Y - ref)) <= \
                1e-13 * numpy.max(numpy.abs(ref))
    finally:
        for h in (hab, h1, h2, hb):
            gpu_lib.slq_op_destroy(h)


def test_cost_of_a_long_row(gpu_lib):
    # a full row last in its tile takes no longer than first in it: searched
    # for in the fifteen others by one wavefront, it took 14 times as long
    n = 65536

    def best(row):
        E = scipy.sparse.csr_matrix(
            (numpy.full(n, 1e-6), (numpy.full(n, row), numpy.arange(n))),
            shape=(n, n))
        A = (scipy.sparse.diags([4.0, 0.5, 0.5], [0, 1, -1], shape=(n, n)) +
             E).tocsr()
        A.sort_indices()
        times = []
        for _ in range(5):
            t0 = time.perf_counter()
            h = _handle(gpu_lib, A.shape, A.indptr, A.indices, A.data)
            times.append(time.perf_counter() - t0)
            gpu_lib.slq_op_destroy(h)
        return min(times)
    assert best(15) <= 3.0 * best(0)
