"""The second Gram-Schmidt pass, which runs only where the first cancels:
matrices of a few distinct eigenvalues, whose residual vanishes after as many
steps while the recurrence is told to go on, so that only an orthogonal basis
keeps the later coefficients harmless."""

import ctypes

import numpy
import pytest
import scipy.sparse

import imate_amd
from imate_amd import _lib

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
