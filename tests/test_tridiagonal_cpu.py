"""The device's tridiagonal eigensolver (imate_amd/csrc/dc.hpp) built for the
host, one thread, against numpy's dense eigensolver; the host path's
quadrature (imate_amd/csrc/ql.hpp) of nodes without weight."""

import ctypes
import os
import subprocess

import numpy
import pytest

from imate_amd import _lib

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
EPS = numpy.finfo(float).eps


@pytest.fixture(scope='module')
def host(tmp_path_factory):
    out = str(tmp_path_factory.mktemp('host') / 'tridiagonal.so')
    subprocess.check_call([
        'g++', '-O2', '-std=c++17', '-fPIC', '-shared',
        '-I' + os.path.join(ROOT, 'imate_amd', 'csrc'),
        '-I' + os.path.join(ROOT, 'include'), '-o', out,
        os.path.join(HERE, 'tridiagonal_host.cpp')])
    return ctypes.CDLL(out)


@pytest.fixture
def solve(host):
    def run(d, e):
        K = len(d)
        d = numpy.ascontiguousarray(d, dtype=float)
        e = numpy.ascontiguousarray(e, dtype=float)
        theta, first = numpy.zeros(K), numpy.zeros(K)
        args = [x.ctypes.data_as(ctypes.c_void_p) for x in (d, e)]
        outs = [x.ctypes.data_as(ctypes.c_void_p) for x in (theta, first)]
        return bool(host.divide_and_conquer(*args, K, *outs)), theta, first
    return run


def _check(solve, d, e):
    """Eigenvalues and weighted moments to a few eps of the norm (weights of
    close nodes are shared arbitrarily)."""
    K = len(d)
    scale = max(numpy.max(numpy.abs(d)), numpy.max(numpy.abs(e[:K - 1]),
                                                   initial=0.0))
    a, b = d / scale, e[:K - 1] / scale
    w, U = numpy.linalg.eigh(numpy.diag(a) + numpy.diag(b, 1) +
                             numpy.diag(b, -1))
    ok, theta, first = solve(d, e)
    assert ok
    t = theta / scale
    tol = 8 * EPS * (8 + numpy.sqrt(K))
    assert numpy.max(numpy.abs(numpy.sort(t) - w)) <= tol
    for p in range(4):
        got, want = numpy.sum(first**2 * t**p), numpy.sum(U[0]**2 * w**p)
        assert abs(got - want) <= tol * 3.0**p


@pytest.mark.parametrize('coupling', [
    1e-100, 1e-150, 1e-161, 1e-163, 1e-200, 1e-300, 5e-324])
def test_negligible_couplings(solve, coupling):
    # equal diagonals: the rotation of a 2 x 2 block is coupling / |coupling|
    for d in ([1.0, 1.0], [1e-3, 1e-3], [1.0] * 5,
              [0.0, 0.0, 0.0, 0.0, 1.0, 2.0]):
        K = len(d)
        _check(solve, numpy.array(d), numpy.full(K, coupling))
        # merges of blocks of mixed sizes
        e = numpy.where(numpy.arange(K) % 2, 0.5, coupling)
        _check(solve, numpy.array(d), e)
        _check(solve, numpy.array(d), e[::-1].copy())


@pytest.mark.parametrize('lowest', [-5, -100, -160, -200, -320])
def test_random_magnitudes(solve, lowest):
    rng = numpy.random.default_rng(-lowest)
    for _ in range(300):
        K = int(rng.integers(2, 34))
        d, e = (10.0**rng.uniform(lowest, 0, K) * rng.choice([-1, 1], K)
                for _ in range(2))
        d[rng.random(K) < 0.3] = 0.0
        d[0] = 1.0
        e[rng.random(K) < 0.3] = 0.0
        _check(solve, d, e)


def test_largest_and_smallest_magnitudes(solve):
    # finite entries whose moduli sum to more than the largest double, and
    # entries near the smallest
    for K in (2, 3, 5, 20, 33):
        for scale in (8e307, 1e-280):
            _check(solve, numpy.full(K, scale), numpy.full(K, 0.5 * scale))
            d = numpy.full(K, 1.5 * scale)
            d[::2] = -scale
            _check(solve, d, numpy.full(K, 0.1 * scale))
    for bad in (numpy.nan, numpy.inf, -numpy.inf):
        for at in (0, 2, 4):
            d = numpy.ones(5)
            d[at] = bad
            assert not solve(d, numpy.ones(5))[0]
            if at < 4:
                assert not solve(numpy.ones(5), d)[0]


def _host_sum(host, alpha, beta, func, gram=0, coefficient=0.0):
    host.quadrature.restype = ctypes.c_double
    args = [numpy.ascontiguousarray(x, dtype=float) for x in (alpha, beta)]
    return host.quadrature(*[x.ctypes.data_as(ctypes.c_void_p) for x in args],
                           len(alpha), gram, func,
                           ctypes.c_double(coefficient))


@pytest.mark.parametrize('gram', [0, 1])
@pytest.mark.parametrize('func,want', [(_lib.FUNC_LOG, numpy.log),
                                       (_lib.FUNC_INV, lambda x: 1.0 / x)])
def test_nodes_of_zero_weight(host, gram, func, want):
    # the second entry is out of the probe's reach and singular
    alpha, beta = numpy.array([2.0, 0.0, 3.0]), numpy.zeros(3)
    got = _host_sum(host, alpha, beta, func, gram)
    assert abs(got - want(4.0 if gram else 2.0)) <= 4 * EPS


def test_weights_at_the_rounding_level(host):
    # the second node is -9e-32 with tau = 3e-16: log of it is NaN
    assert _host_sum(host, [1.0, 0.0], [3e-16, 0.0], _lib.FUNC_LOG) == 0.0
    # a node of real weight keeps its NaN
    assert numpy.isnan(_host_sum(host, [1.0, 0.0], [1e-6, 0.0],
                                 _lib.FUNC_LOG))


@pytest.mark.parametrize('k', [1, 2, 3, 8, 20, 33])
@pytest.mark.parametrize('low', [0.0, 1e-17, 1e-9, 0.5])
def test_zero_singular_values(host, k, low):
    # exp(-sigma^2) is 1 at a zero singular value, whose weight the two
    # eigenvectors of the Golub-Kahan tridiagonal share arbitrarily
    rng = numpy.random.default_rng(k)
    tol = 8 * EPS * (8 + numpy.sqrt(2 * k))
    for at in {0, k // 2, k - 1}:
        alpha, beta = 1.0 + rng.random(k), 0.3 + 0.5 * rng.random(k)
        alpha[at] = low
        _, s, vt = numpy.linalg.svd(numpy.diag(alpha) +
                                    numpy.diag(beta[:k - 1], 1))
        want = numpy.sum(vt[:, 0]**2 * numpy.exp(-s**2))
        got = _host_sum(host, alpha, beta, _lib.FUNC_EXP, 1, -1.0)
        assert abs(got - want) <= tol * max(1.0, s[0]**2)
