"""GPU: average and standard deviation where the sums about the first value
cancel: a small spread far from zero, a first value far from all others, a
constant. Reference: exact sums of rationals. The deviations d = x - x0 carry
2^-53 of themselves, so the standard deviation is off by at most 2^-53 times
rms(d) / std, and by the few roundings after the sums."""
from fractions import Fraction
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _values(kind, n, rng):
    if kind == 'constant':
        return np.full(n, 1. / 3.)
    v = rng.random(n) * (1e-3 if kind == 'offset' else 1.) + (1e6 if kind == 'offset' else 1.)
    if kind == 'outlier':
        v[0] = 1e8
    return v


@pytest.mark.parametrize('real', ['double', 'float'])
@pytest.mark.parametrize('size', [(37,), (70, 33), (301, 233)])
@pytest.mark.parametrize('kind', ['offset', 'outlier', 'constant', 'plain'])
def test_shifted_sums(real, size, kind):
    from hydro.solver.hipfvsolver import HipFVSolver
    s = HipFVSolver(dim=len(size), gridSize=size, integrator='forward Euler', boundary='periodic', real=real)
    n = math.prod(size)
    v = _values(kind, n, np.random.default_rng(n)).astype(s.dtype)
    U = np.zeros(s.shape, s.dtype)
    U[..., 0] = 1
    U[..., 4] = 1e3
    inner = (0, slice(2, -2) if len(size) > 1 else 0, slice(2, -2))
    U[inner + (0,)] = v.reshape(size[::-1])
    s.resetState(U)
    mn, mx, avg, std = s.calcDisplayVarRangeAndAvgAndStdDev(0)
    x = [Fraction(float(a)) for a in v]
    mean = sum(x) / n
    var = sum((a - mean) ** 2 for a in x) / n
    assert mn == v.min() and mx == v.max()
    assert abs(avg - float(mean)) <= 2 ** -52 * abs(float(mean))
    ref = math.sqrt(var)
    rms = math.sqrt(sum((a - x[0]) ** 2 for a in x) / n)
    assert abs(std - ref) <= 2 ** -53 * (rms + 8 * ref)
