"""The second Gram-Schmidt pass, which runs only where the first cancels: the
remainder it leaves where nothing is left of a residual, the coefficients of
runs that take it in every step, and its cost. (The samples of runs that go on
past an invariant subspace hardly depend on it: the couplings there are at the
rounding level, so the later coefficients weigh nothing.)"""

import os
import time

import numpy
import pytest
import scipy.sparse

import imate_amd
from imate_amd import _lib
from imate_amd.linear_operator import Matrix

pytestmark = pytest.mark.gpu


def _probes(seed, n, count):
    X = numpy.empty((count, n))
    _lib.check(_lib.load().slq_rademacher(
        seed, n, 0, count, _lib.SLQ_F64, _lib.ptr(X), None), 'slq_rademacher')
    return X


def _few_eigenvalues(n, values, seed):
    """Block-diagonal symmetric matrix of 4 x 4 blocks with the eigenvalues
    drawn from ``values``."""
    rng = numpy.random.default_rng(seed)
    blocks = []
    for _ in range(0, n, 4):
        Q, _ = numpy.linalg.qr(rng.standard_normal((4, 4)))
        blocks.append(Q @ numpy.diag(rng.choice(values, 4)) @ Q.T)
    A = scipy.sparse.block_diag(blocks, format='csr')
    A = (A + A.T) * 0.5
    return A.tocsr()


# 30 and 45 steps take more than 8, 16 and 32 vectors a pass; 24 samples
# leave 40 lanes without a probe
@pytest.mark.parametrize('m', [12, 30, 45])
@pytest.mark.parametrize('samples', [64, 24])
def test_lanczos_goes_on_past_an_invariant_subspace(gpu_lib, m, samples):
    n, values = 400, [0.5, 1.0, 1.7, 2.5, 4.0]
    A = _few_eigenvalues(n, values, 3)
    _, info = imate_amd.logdet(
        A, method='slq', gpu=True, lanczos_degree=m, lanczos_tol=1e-300,
        min_num_samples=samples, max_num_samples=samples, seed=9,
        orthogonalize=-1, error_rtol=0.0, return_info=True)
    got = numpy.asarray(info['convergence']['samples'])
    w, U = numpy.linalg.eigh(A.toarray())
    Z = _probes(9, n, samples)
    want = ((Z @ U)**2) @ numpy.log(w)
    # the exact value from step 5 on; the junk couplings are of size eps
    assert numpy.max(numpy.abs(got - want)) <= 1e-10 * numpy.max(
        numpy.abs(want))


@pytest.mark.parametrize('m', [10, 20])
def test_golub_kahn_goes_on_past_an_invariant_subspace(gpu_lib, m):
    n = 400
    A = _few_eigenvalues(n, [0.8, 1.0, 1.5, 2.0], 4)
    _, info = imate_amd.logdet(
        A, gram=True, method='slq', gpu=True, lanczos_degree=m,
        lanczos_tol=1e-300, min_num_samples=32, max_num_samples=32, seed=9,
        orthogonalize=-1, error_rtol=0.0, return_info=True)
    got = numpy.asarray(info['convergence']['samples'])
    w, U = numpy.linalg.eigh((A.T @ A).toarray())
    Z = _probes(9, n, 32)
    want = ((Z @ U)**2) @ numpy.log(w)
    assert numpy.max(numpy.abs(got - want)) <= 1e-10 * numpy.max(
        numpy.abs(want))


def _recurrences(A, m, samples=64, gram=0, mode=None):
    """alpha, beta [samples, m] of the re-orthogonalised recurrence, with
    SLQ_FUSED_GS = mode."""
    M = Matrix(A)
    handle = M.get_linear_operator(gpu=True).handle
    alpha = numpy.zeros((samples, m))
    beta = numpy.zeros((samples, m))
    sizes = numpy.zeros(samples, dtype=numpy.int32)
    keep = os.environ.pop('SLQ_FUSED_GS', None)
    if mode is not None:
        os.environ['SLQ_FUSED_GS'] = str(mode)
    try:
        _lib.check(_lib.load().slq_recurrences(
            handle, 0.0, gram, 9, 0, samples, m, 1e-300, -1, 0,
            _lib.ptr(alpha), _lib.ptr(beta), _lib.ptr(sizes)),
            'slq_recurrences')
    finally:
        os.environ.pop('SLQ_FUSED_GS', None)
        if keep is not None:
            os.environ['SLQ_FUSED_GS'] = keep
    return alpha, beta


def _tridiagonal(n, seed):
    rng = numpy.random.default_rng(seed)
    off = -0.3 - 0.2 * rng.random(n - 1)
    return scipy.sparse.diags([2.0 + rng.random(n), off, off], [0, 1, -1],
                              format='csr')


# a basis of 8, 16, 32, 64 and more vectors: every form of the first pass
@pytest.mark.parametrize('samples', [64, 24])
@pytest.mark.parametrize('n', [8, 16, 20, 32, 45, 64, 65, 70])
def test_remainder_where_nothing_is_left(gpu_lib, n, samples):
    # the last step's residual lies in the span of the n basis vectors but
    # for rounding: it is 3e-15 and more without a pass, 3e-32 and more after
    # one, below 3e-46 after two (FP64, such matrices of 8 to 70 rows)
    _, beta = _recurrences(_tridiagonal(n, n), n, samples)
    assert numpy.all(beta[:, :-1] > 1e-9)
    assert numpy.max(beta[:, -1]) < 1e-40


# many workgroups, every form; in numpy the coefficients of one and two passes
# agree to 3e-15. Golub-Kahn leaves the oldest vector out of its window, and
# rounding along that vector grows fourfold a step: 4e-16 up to step 25 and
# 1e-8 at step 40, in numpy too, so it is compared over 24 steps
@pytest.mark.parametrize('gram,m', [(0, 70), (1, 24)])
@pytest.mark.parametrize('n,samples', [(3001, 64), (20011, 24)])
def test_second_pass_in_every_step(gpu_lib, gram, m, n, samples):
    A = _tridiagonal(n, 5)
    plain = _recurrences(A, m, samples, gram, mode=0)
    for mode in (None, 2):
        got = _recurrences(A, m, samples, gram, mode)
        for x, y in zip(got, plain):
            assert numpy.max(numpy.abs(x - y)) <= 1e-12


@pytest.mark.parametrize('n,m', [(2000, 60), (2000, 80)])
def test_cost_of_the_second_pass(gpu_lib, n, m):
    # Golub-Kahn on 11 distinct values: every step past the eleventh cancels.
    # Its products come from the first subtraction's read of the basis (up to
    # 64 vectors) and its totals from all workgroups, so that it takes less
    # than separate passes; a total in one workgroup took six times as long
    A = scipy.sparse.diags(1.0 + numpy.arange(n) % 11, format='csr')
    M = Matrix(A)

    def best(mode):
        os.environ['SLQ_FUSED_GS'] = str(mode)
        times = []
        for _ in range(6):
            t0 = time.perf_counter()
            imate_amd.logdet(M, gram=True, method='slq', gpu=True,
                             lanczos_degree=m, min_num_samples=64,
                             max_num_samples=64, orthogonalize=-1, seed=1)
            times.append(time.perf_counter() - t0)
        return min(times)
    keep = os.environ.pop('SLQ_FUSED_GS', None)
    try:
        separate, fused = best(0), best(1)
    finally:
        os.environ.pop('SLQ_FUSED_GS', None)
        if keep is not None:
            os.environ['SLQ_FUSED_GS'] = keep
    assert fused <= 1.5 * separate
