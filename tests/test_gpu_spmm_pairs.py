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
