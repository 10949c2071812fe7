"""Dot products (the reductions' wave sums) at lengths around a lane, a wave and
a block, against exact summation: the error of any summation order of n
products is at most n eps sum |a_i b_i|.  Infinities and NaN pass through."""
import math

import numpy as np
import pytest

import multiscalefemsolver3d_amd as mfs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 31, 33, 63, 64, 65, 255, 257, 1025, 100_003])
def test_dot_error_bound(ctx, n):
    g = np.random.default_rng(n)
    a, b = g.normal(size=n), g.normal(size=n) * np.exp(g.uniform(-8, 8, n))
    d = mfs.dot(mfs.Vec(ctx, n, mfs.F64, a), mfs.Vec(ctx, n, mfs.F64, b))
    assert abs(d - math.fsum(a * b)) <= 2 * n * np.finfo(float).eps * np.abs(a * b).sum()
    for lane in {0, n // 2, n - 1}:  # each lane reaches the sum
        e = np.zeros(n)
        e[lane] = 3.0
        assert mfs.dot(mfs.Vec(ctx, n, mfs.F64, e), mfs.Vec(ctx, n, mfs.F64, a)) == 3.0 * a[lane]
        e[lane] = np.inf
        assert mfs.dot(mfs.Vec(ctx, n, mfs.F64, e), mfs.Vec(ctx, n, mfs.F64, np.ones(n))) == np.inf
        e[lane] = np.nan
        assert math.isnan(mfs.dot(mfs.Vec(ctx, n, mfs.F64, e), mfs.Vec(ctx, n, mfs.F64, np.ones(n))))
