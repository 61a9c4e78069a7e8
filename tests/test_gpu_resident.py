"""Lanczos of small matrices in one launch against the block kernels (asked
for with a launch setting) on the same probes: recurrence coefficients at the
sizes where lanes, rounds and threads change, every operand type, the shift,
an early breakdown; and a dispatch that a long row takes back."""

import ctypes

import numpy
import pytest
import scipy.sparse

from imate_amd import _lib

pytestmark = pytest.mark.gpu


def _spd(n, k, seed, dtype='float64'):
    """Band of about k entries a row, diagonally dominant."""
    rng = numpy.random.default_rng(seed)
    h = max(0, min(n - 1, (k - 1) // 2))
    d = [rng.uniform(-1.0, 1.0, n - i) for i in range(1, h + 1)]
    A = scipy.sparse.diags(d, range(1, h + 1), shape=(n, n)) if h else \
        scipy.sparse.csr_matrix((n, n))
    A = A + A.T + scipy.sparse.diags(rng.uniform(1.2, 2.0, n) * (k + 1))
    A = A.tocsr().astype(dtype)
    A.sort_indices()
    return A


def _handle(lib, A):
    ip = numpy.ascontiguousarray(A.indptr, dtype=numpy.int64)
    h = ctypes.c_void_p()
    _lib.check(lib.slq_op_create_csr(
        A.shape[0], A.shape[1], A.nnz, _lib.ptr(ip),
        _lib.ptr(numpy.ascontiguousarray(A.indices, dtype=numpy.int32)),
        _lib.ptr(A.data), _lib.dtype_code(A.dtype), ctypes.byref(h)),
        'slq_op_create_csr')
    return h


def _recurrences(lib, h, m, count=64, t=0.0, precision=0, tol=1e-14):
    al = numpy.zeros((count, m))
    be = numpy.zeros((count, m))
    sz = numpy.zeros(count, dtype=numpy.int32)
    _lib.check(lib.slq_recurrences(h, t, 0, 5, 0, count, m, tol, 0, precision,
                                   _lib.ptr(al), _lib.ptr(be), _lib.ptr(sz)),
               'slq_recurrences')
    return al, be, sz


def _both(lib, h, m, **kw):
    a = _recurrences(lib, h, m, **kw)
    _lib.check(lib.slq_op_set_launch(h, 0, 0, 1, 0), 'slq_op_set_launch')
    b = _recurrences(lib, h, m, **kw)
    _lib.check(lib.slq_op_set_launch(h, 0, 0, 0, 0), 'slq_op_set_launch')
    return a, b


# 4, 8, 16 and 32 lanes a row; 128 / 129 threads; partly filled rounds
@pytest.mark.parametrize('n,k', [
    (1, 1), (2, 1), (5, 3), (63, 3), (64, 7), (65, 13), (128, 27), (129, 27),
    (130, 59), (255, 3), (257, 13), (513, 13), (700, 27), (1000, 47),
    (1025, 3), (300, 75), (5000, 3)])
@pytest.mark.parametrize('dtype', ['float64', 'float32'])
def test_coefficients_equal_block_kernels(gpu_lib, n, k, dtype):
    A = _spd(n, k, n + k, dtype)
    h = _handle(gpu_lib, A)
    try:
        m = min(6, n)
        (a1, b1, s1), (a2, b2, s2) = _both(gpu_lib, h, m)
        # six steps amplify rounding by little on these matrices
        tol = 1e-11 if dtype == 'float64' else 2e-5
        scale = numpy.max(numpy.abs(a2))
        assert numpy.array_equal(s1, s2)
        if dtype == 'float32' and n >= 63:
            # two kernels: the resident one keeps FP64 vectors
            assert not numpy.array_equal(a1, a2)
        for p in range(64):
            q = s1[p]
            assert numpy.max(numpy.abs(a1[p, :q] - a2[p, :q])) <= tol * scale
            assert numpy.max(numpy.abs(b1[p, :q] - b2[p, :q])) <= tol * scale
        if dtype == 'float64':
            (a1, _, _), (a2, _, _) = _both(gpu_lib, h, m, precision=1)
            assert numpy.max(numpy.abs(a1[:, 0] - a2[:, 0])) <= 2e-5 * scale
    finally:
        gpu_lib.slq_op_destroy(h)


@pytest.mark.parametrize('count', [64, 23])
def test_shift_and_partial_block(gpu_lib, count):
    A = _spd(400, 9, 1)
    ha = _handle(gpu_lib, A)
    h = ctypes.c_void_p()
    _lib.check(gpu_lib.slq_op_create_affine(ha, None, ctypes.byref(h)),
               'slq_op_create_affine')
    try:
        (a1, b1, s1), (a2, b2, s2) = _both(gpu_lib, h, 8, t=0.75, count=count)
        scale = numpy.max(numpy.abs(a2))
        assert numpy.max(numpy.abs(a1 - a2)) <= 1e-11 * scale
        assert numpy.max(numpy.abs(b1 - b2)) <= 1e-11 * scale
    finally:
        gpu_lib.slq_op_destroy(h)
        gpu_lib.slq_op_destroy(ha)


def test_breakdown_ends_the_recurrence(gpu_lib):
    n = 96
    A = scipy.sparse.diags(numpy.where(numpy.arange(n) % 3 == 0, 1.0,
                                       numpy.where(numpy.arange(n) % 3 == 1,
                                                   2.0, 5.0))).tocsr()
    h = _handle(gpu_lib, A)
    try:
        (a1, b1, s1), (a2, b2, s2) = _both(gpu_lib, h, 10, tol=1e-12)
        assert numpy.all(s1 == 3) and numpy.array_equal(s1, s2)
        assert numpy.max(numpy.abs(a1[:, :3] - a2[:, :3])) <= 1e-11
    finally:
        gpu_lib.slq_op_destroy(h)


def test_long_row_keeps_the_block_kernels(gpu_lib):
    """An arrow matrix: one full row among short ones."""
    n = 4000
    A = scipy.sparse.lil_matrix((n, n))
    A.setdiag(numpy.linspace(2.0, 3.0, n))
    A[0, :] = 1e-3
    A[:, 0] = 1e-3
    A[0, 0] = 5.0
    A = A.tocsr()
    h = _handle(gpu_lib, A)
    try:
        (a1, b1, _), (a2, b2, _) = _both(gpu_lib, h, 5)
        assert numpy.array_equal(a1, a2) and numpy.array_equal(b1, b2)
    finally:
        gpu_lib.slq_op_destroy(h)
