"""Training kernels of the surrogate MLP at the edges of their sample tiles
and work split: gradients against the CPU oracle, and the same training
whether its steps are replayed from a graph or launched."""

import ctypes

import numpy
import pytest

from imate_amd import _lib
from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu

f32 = numpy.float32


def _data(B, seed):
    rng = numpy.random.default_rng(seed)
    x = rng.uniform(-1, 1, (B, 2)).astype(f32)
    return x, (numpy.sin(2 * x[:, 0]) + x[:, 1] ** 2).astype(f32)


# one tile has 16 samples; 128 tiles are the last with a workgroup each, 512
# the last with two per workgroup
@pytest.mark.parametrize('B', [15, 16, 17, 2048, 2049, 8192, 8193])
def test_gradient_at_tile_edges(gpu_lib, B):
    p = M.init(3).astype(f32)
    x, t = _data(B, B)
    g = numpy.full(M.NUM_PARAMS, numpy.nan, dtype=f32)
    loss = ctypes.c_float(0)
    _lib.check(gpu_lib.slq_mlp_grad(_lib.ptr(p), _lib.ptr(x), _lib.ptr(t), B,
                                    ctypes.byref(loss), _lib.ptr(g)), 'grad')
    args = [a.astype(numpy.float64) for a in (p, x, t)]
    gr, lr = M.grad(*args), M.loss(*args)
    assert abs(loss.value - lr) <= 1e-5 * lr
    for lo, hi in [(0, 256), (256, 384), (384, 16768), (16768, 16896),
                   (16896, 17024), (17024, 17025)]:
        scale = numpy.abs(gr[lo:hi]).max()
        assert numpy.abs(g[lo:hi] - gr[lo:hi]).max() <= 2e-5 * scale + 1e-9, (lo, hi)


# 31 steps are launched one by one, 32 and 37 replay a graph of 16 twice
@pytest.mark.parametrize('steps', [32, 37])
def test_replayed_steps_equal_launched_ones(gpu_lib, steps):
    x, t = _data(100, 5)
    losses = {}
    for k in (31, steps):
        p = M.init(7).astype(f32)
        losses[k] = numpy.full(k, numpy.nan, dtype=f32)
        _lib.check(gpu_lib.slq_mlp_train(_lib.ptr(p), _lib.ptr(x), _lib.ptr(t), 100, k,
                                         f32(1e-3), _lib.ptr(losses[k])), 'train')
    assert numpy.array_equal(losses[31], losses[steps][:31])
    assert numpy.isfinite(losses[steps]).all()
