"""Matrix-core SpMM at the lengths of a tile's slab list where its loops hand
over: one to a few times the three pairs of four-slab groups in flight, and
one past them, against scipy in FP64. Also with the looping form of a capped
grid, which must give the same bits."""

import ctypes

import numpy
import pytest
import scipy.sparse

from imate_amd import _lib

pytestmark = pytest.mark.gpu


# columns of a tile; eight to a pair
@pytest.mark.parametrize('c', [1, 8, 9, 16, 17, 24, 25, 32, 33, 40, 41, 48, 49, 56, 57, 97])
@pytest.mark.parametrize('dtype', [numpy.float64, numpy.float32])
def test_product(gpu_lib, c, dtype):
    nrows, ncols = 16 * 19 + 5, 400
    rng = numpy.random.default_rng(c)
    cols = [numpy.sort(rng.choice(ncols, c, replace=False)) for _ in range(20)]
    indices = numpy.concatenate([cols[i // 16] for i in range(nrows)]).astype(numpy.int32)
    data = rng.standard_normal(nrows * c).astype(dtype)
    ip = numpy.arange(nrows + 1, dtype=numpy.int64) * c
    A = scipy.sparse.csr_matrix((data, indices, ip), shape=(nrows, ncols))
    X = rng.standard_normal((ncols, 64)).astype(dtype)
    h = ctypes.c_void_p()
    _lib.check(gpu_lib.slq_op_create_csr(
        nrows, ncols, A.nnz, _lib.ptr(ip), _lib.ptr(indices), _lib.ptr(data),
        _lib.dtype_code(dtype), ctypes.byref(h)), 'create')
    try:
        Y = [numpy.full((nrows, 64), numpy.nan, dtype=dtype) for _ in range(2)]
        for y, grid in zip(Y, (0, 1)):
            _lib.check(gpu_lib.slq_op_set_launch(h, grid, 0, 0, 0), 'set_launch')
            _lib.check(gpu_lib.slq_op_spmm(h, 0.0, 64, 0, _lib.ptr(X), _lib.ptr(y)),
                       'slq_op_spmm')
        # c products summed: c eps of the sum of moduli
        bound = c * numpy.finfo(dtype).eps * (
            abs(A).astype(numpy.float64) @ numpy.abs(X.astype(numpy.float64)))
        ref = A.astype(numpy.float64) @ X.astype(numpy.float64)
        assert numpy.all(numpy.abs(Y[0] - ref) <= bound)
        assert numpy.array_equal(Y[0], Y[1])
    finally:
        gpu_lib.slq_op_destroy(h)


# 256 partial rows of 128 matrix rows are added in one launch, more in two
@pytest.mark.parametrize('n', [32640, 32768, 32770, 33800, 66000])
def test_total_over_the_tiles(gpu_lib, n):
    d = numpy.random.default_rng(n).random(n)
    A = scipy.sparse.diags([2.0 + d] + [-0.1] * 16,
                           list(range(0, 9)) + list(range(-8, 0)),
                           shape=(n, n), format='csr')
    h = ctypes.c_void_p()
    ip = A.indptr.astype(numpy.int64)
    _lib.check(gpu_lib.slq_op_create_csr(
        n, n, A.nnz, _lib.ptr(ip), _lib.ptr(A.indices), _lib.ptr(A.data),
        _lib.SLQ_F64, ctypes.byref(h)), 'create')
    Z = numpy.empty((64, n))
    _lib.check(gpu_lib.slq_rademacher(5, n, 0, 64, _lib.SLQ_F64, _lib.ptr(Z),
                                      None), 'slq_rademacher')
    alpha, beta = numpy.zeros((64, 1)), numpy.zeros((64, 1))
    sizes = numpy.zeros(64, dtype=numpy.int32)
    try:
        _lib.check(gpu_lib.slq_recurrences(
            h, 0.0, 0, 5, 0, 64, 1, 1e-14, 0, 0, _lib.ptr(alpha),
            _lib.ptr(beta), _lib.ptr(sizes)), 'slq_recurrences')
        want = numpy.einsum('pi,pi->p', Z, (A @ Z.T).T) / n
        # sums of n terms of size 1/n, added in parts of 128 rows
        assert numpy.max(numpy.abs(alpha[:, 0] - want)) <= 1e-13
    finally:
        gpu_lib.slq_op_destroy(h)
