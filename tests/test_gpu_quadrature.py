"""Device eigensolve and quadrature (slq_quadrature) against numpy's dense
eigensolver / SVD: sizes around the wavefront, the two solvers and the
inquiry counts; deflating, zero and non-finite matrices."""

import numpy
import pytest

from imate_amd import _lib

pytestmark = pytest.mark.gpu

EPS = numpy.finfo(float).eps


def _run(alpha, beta, sizes, gram=0, func=_lib.FUNC_IDENT, params=None,
         n=1.0, coefficients=None):
    lib = _lib.load()
    count, m = alpha.shape
    q = 1 if params is None else len(params)
    samples = numpy.zeros((count, q))
    theta = numpy.zeros((count, m))
    tau = numpy.zeros((count, m))
    sz = numpy.asarray(sizes, dtype=numpy.int32)
    _lib.check(lib.slq_quadrature(
        _lib.ptr(alpha), _lib.ptr(beta), _lib.ptr(sz), count, m, gram, func,
        _lib.ptr(coefficients), 1.0, n, _lib.ptr(params), q, 0 if params is None else 1,
        _lib.ptr(samples), _lib.ptr(theta), _lib.ptr(tau)), 'slq_quadrature')
    return samples, theta, tau


def _dense(a, b, gram):
    k = len(a)
    T = numpy.diag(a) + numpy.diag(b[:k - 1], 1)
    if gram:
        # T is the bidiagonal: right singular vectors of it
        _, s, vt = numpy.linalg.svd(T)
        return s**2, vt[:, 0]
    T += numpy.diag(b[:k - 1], -1)
    w, U = numpy.linalg.eigh(T)
    return w, U[0]


# 32/33, 64/65, 128/129: thread counts; 512/513 (gram) and 1024/1025: the last
# divide-and-conquer size and the first of the serial solver
@pytest.mark.parametrize('gram,m', [
    (0, 1), (0, 2), (0, 3), (0, 20), (0, 31), (0, 32), (0, 33), (0, 64),
    (0, 65), (0, 128), (0, 129), (0, 200),
    (0, 1024), (0, 1025), (1, 1), (1, 2), (1, 16), (1, 32), (1, 33), (1, 60),
    (1, 512), (1, 513)])
def test_nodes_and_weights(gram, m):
    rng = numpy.random.default_rng(m)
    count = 3
    alpha = 2.0 + rng.random((count, m))
    beta = 0.2 + 0.5 * rng.random((count, m))
    # probe 1 ends early; probe 2 nearly decouples (deflation)
    sizes = [0, max(1, m // 2), 0]
    beta[2, ::3] *= 1e-14
    q = numpy.array([0.0, 0.5])
    samples, theta, tau = _run(alpha, beta, sizes, gram, n=10.0)
    shifted, _, _ = _run(alpha, beta, sizes, gram, _lib.FUNC_INV, q, n=10.0)
    for p in range(count):
        k = sizes[p] or m
        w, z = _dense(alpha[p, :k], beta[p, :k], gram)
        order = numpy.argsort(theta[p, :k])
        norm = numpy.max(w)
        # backward error of either solver: a few eps |T| per level / sweep
        tol = 8 * EPS * (8 + numpy.sqrt(k))
        assert numpy.max(numpy.abs(theta[p, :k][order] - numpy.sort(w))) \
            <= tol * norm
        assert abs(numpy.sum(tau[p, :k]**2) - 1.0) <= tol
        assert numpy.all(theta[p, k:] == 0.0)
        # sums over nodes: weights of close nodes are shared arbitrarily
        assert abs(samples[p, 0] - 10.0 * numpy.sum(z**2 * w)) \
            <= 10.0 * tol * norm
        low = numpy.min(w)
        for j in range(2):
            want = 10.0 * numpy.sum(z**2 / (w + q[j]))
            assert abs(shifted[p, j] - want) <= \
                10.0 * tol * norm / (low + q[j])**2


@pytest.mark.parametrize('q', [1, 8, 9, 64, 65, 300])
@pytest.mark.parametrize('m', [17, 70])
def test_many_inquiries(q, m):
    rng = numpy.random.default_rng(q)
    alpha = 2.0 + rng.random((64, m))
    beta = 0.2 + 0.5 * rng.random((64, m))
    t = numpy.linspace(0.0, 3.0, q) + 0.25
    samples, _, _ = _run(alpha, beta, numpy.zeros(64), 0, _lib.FUNC_LOG, t,
                         n=7.0)
    for p in (0, 63):
        w, z = _dense(alpha[p], beta[p], 0)
        want = [7.0 * numpy.sum(z**2 * numpy.log(w + x - t[0])) for x in t]
        assert numpy.max(numpy.abs(samples[p] - want)) < 1e-12


def test_scaled_zero_and_non_finite():
    m = 6
    alpha = numpy.ones((5, m))
    beta = numpy.full((5, m), 0.25)
    alpha[1] *= 1e150
    beta[1] *= 1e150
    alpha[2] = 0.0
    beta[2] = 0.0
    alpha[3, 2] = numpy.nan
    beta[4, 1] = numpy.inf
    samples, theta, _ = _run(alpha, beta, numpy.zeros(5))
    assert abs(samples[0, 0] - 1.0) < 1e-14
    assert abs(samples[1, 0] - 1e150) < 1e136
    assert samples[2, 0] == 0.0
    assert numpy.isnan(samples[3, 0]) and numpy.isnan(samples[4, 0])


@pytest.mark.parametrize('coupling', [1e-161, 1e-163, 1e-300])
def test_couplings_whose_squares_underflow(coupling):
    # equal diagonals, as a Lanczos run on a multiple of the identity gives
    for m in (2, 3, 20):
        alpha = numpy.full((1, m), 2.0)
        beta = numpy.full((1, m), coupling)
        samples, theta, tau = _run(alpha, beta, [0])
        assert numpy.all(theta == 2.0)
        tol = 8 * EPS * (8 + numpy.sqrt(m))
        assert abs(numpy.sum(tau**2) - 1.0) <= tol
        assert abs(samples[0, 0] - 2.0) <= 2.0 * tol


def test_finite_entries_whose_sum_overflows():
    m = 20
    alpha = numpy.full((1, m), 1.5e308)
    beta = numpy.full((1, m), 1e307)
    w, z = _dense(numpy.full(m, 1.5), numpy.full(m, 0.1), 0)
    _, theta, tau = _run(alpha, beta, [0])
    tol = 8 * EPS * (8 + numpy.sqrt(m))
    assert numpy.max(numpy.abs(numpy.sort(theta[0]) / 1e308 - w)) <= 2 * tol
    assert abs(numpy.sum(tau**2) - 1.0) <= tol


@pytest.mark.parametrize('gram,m', [(0, 3), (0, 1025), (1, 3), (1, 513)])
def test_nodes_of_zero_weight(gram, m):
    # past the first entry a singular part out of the probe's reach, in both
    # solvers
    alpha = numpy.full((1, m), 2.0)
    alpha[0, 1::2] = 0.0
    beta = numpy.zeros((1, m))
    samples, _, _ = _run(alpha, beta, [0], gram, _lib.FUNC_LOG)
    assert abs(samples[0, 0] - numpy.log(4.0 if gram else 2.0)) <= 4 * EPS


def test_weights_at_the_rounding_level():
    # node -beta^2 with tau = beta: log of it is NaN. A weight of 3e-16
    # squared is rounding, one of 1e-6 squared is not
    alpha = numpy.array([[1.0, 0.0], [1.0, 0.0]])
    beta = numpy.array([[3e-16, 0.0], [1e-6, 0.0]])
    samples, _, _ = _run(alpha, beta, [0, 0], 0, _lib.FUNC_LOG)
    assert abs(samples[0, 0]) <= 4 * EPS
    assert numpy.isnan(samples[1, 0])


# both solvers; a zero and a nearly zero singular value
@pytest.mark.parametrize('k', [1, 2, 20, 33, 100, 512, 513])
@pytest.mark.parametrize('low', [0.0, 1e-17, 1e-9])
def test_zero_singular_values(k, low):
    rng = numpy.random.default_rng(k)
    alpha, beta = 1.0 + rng.random((3, k)), 0.3 + 0.5 * rng.random((3, k))
    for p, at in enumerate((0, k // 2, k - 1)):
        alpha[p, at] = low
    samples, theta, tau = _run(alpha, beta, [0, 0, 0], 1, _lib.FUNC_EXP,
                               coefficients=numpy.array([-1.0]))
    tol = 8 * EPS * (8 + numpy.sqrt(2 * k))
    for p in range(3):
        w, z = _dense(alpha[p], beta[p], 1)
        want = numpy.sum(z**2 * numpy.exp(-w))
        assert abs(samples[p, 0] - want) <= tol * max(1.0, numpy.max(w))
        assert abs(numpy.sum(tau[p]**2) - 1.0) <= tol
