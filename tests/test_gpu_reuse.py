"""A solver or a batch that is given a new state after it has run another: what it
computes is what a fresh one computes. The Euler kernels store only the momenta
that a state has (one in 1D, two in 2D, three where any out-of-plane momentum is
not 0), so the buffers hold those of the state before unless they are cleared; the
comparison is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _state(cfg, outOfPlane):
    from hydro.init import euler as ie
    x, y, z = ie.mesh(cfg)
    shape = ie.interior_shape(cfg)
    rho = np.broadcast_to(1 + .2 * np.sin(2 * np.pi * x) * np.cos(np.pi * y), shape)
    v = [.3 + 0 * rho, (.2 if cfg.dim > 1 else 0.) + 0 * rho, 0 * rho]
    if outOfPlane:
        for a in range(cfg.dim, 3):
            v[a] = .1 * (a + 1) + .05 * rho
    return ie.to_ghosted(cfg, ie.cons_from_prim(rho, v, 1. + 0 * rho, 1.4))


def _same(a, b, what):
    assert np.array_equal(a.UBufObj.toCPU(), b.UBufObj.toCPU()), what
    assert np.array_equal(a.conservedTotals(), b.conservedTotals()), what
    for field in (1, 2, 3, 'v y', 'v z', 'EKin', 'P'):
        assert a.calcDisplayVarRangeAndAvgAndStdDev(field) == b.calcDisplayVarRangeAndAvgAndStdDev(field), (what, field)
    assert (a.t, a.dt) == (b.t, b.dt), what


CASES = [(1, (n,), integ) for n in (5, 113, 241, 1000, 20011)
         for integ in ('forward Euler', 'Runge-Kutta 2, TVD', 'Runge-Kutta 3, TVD')]
CASES += [(2, size, integ) for size in ((70, 33), (300, 200)) for integ in ('forward Euler', 'Runge-Kutta 2, TVD')]


@pytest.mark.parametrize('real,fast', [('double', True), ('float', True), ('double', False)])
@pytest.mark.parametrize('dim,size,integ', CASES)
def test_new_state_with_fewer_momenta(dim, size, integ, real, fast):
    from hydro.solver.hipfvsolver import HipFVSolver
    kw = dict(dim=dim, gridSize=size, usePLM='plm cons', slopeLimiter='minmod', integrator=integ, cfl=.3,
              boundary='freeflow', real=real, fastMath=fast)
    for before in (1, 2, 5):
        s = HipFVSolver(**kw)
        s.resetState(_state(s.cfg, True).astype(s.dtype))
        s.update(before)
        assert np.abs(s.UBufObj.toCPU()[..., 3]).max() > 0
        fresh = HipFVSolver(**kw)
        U = _state(s.cfg, False).astype(s.dtype)
        for v in (s, fresh):
            v.resetState(U)
        for steps in (1, 3):
            for v in (s, fresh):
                v.update(steps)
            _same(s, fresh, (before, steps))
            assert s.calcDT() == fresh.calcDT()
        for v in (s, fresh):      # and back to three components
            v.resetState(_state(s.cfg, True).astype(s.dtype))
            v.update(3)
        _same(s, fresh, (before, 'again'))


@pytest.mark.parametrize('integ', ['forward Euler', 'Runge-Kutta 2, TVD'])
@pytest.mark.parametrize('dim,sizes', [(1, [64, 1000]), (2, [(70, 33), (40, 51)])])
def test_batch_new_state_with_fewer_momenta(dim, sizes, integ):
    from hydro._cfg import make_cfg
    from hydro.solver.batch import HipBatch
    kws = [dict(dim=dim, size=n, plm='plm cons', slope_limiter='minmod', integrator=integ, cfl=.3, boundary='freeflow',
                precision='double', fast_math=True) for n in sizes]
    cfgs = [make_cfg(**kw) for kw in kws]
    b, fresh = HipBatch(kws), HipBatch(kws)
    # one grid without out-of-plane momentum runs with one that has it
    for i, c in enumerate(cfgs):
        b.upload(i, _state(c, i == 1))
    b.constrainU()
    b.update(3)
    for v in (b, fresh):
        for i, c in enumerate(cfgs):
            v.upload(i, _state(c, False))
        v.constrainU()
    for steps in (1, 2, 4):
        for v in (b, fresh):
            v.update(steps)
        for i in range(len(kws)):
            assert np.array_equal(b.download(i), fresh.download(i)), (i, steps)


@pytest.mark.parametrize('integ', ['forward Euler', 'Runge-Kutta 2, TVD'])
def test_batch_grid_that_sits_out(integ):
    """an inactive grid keeps its state while the others step, and goes on from it"""
    from hydro._cfg import make_cfg
    from hydro.solver.batch import HipBatch
    kws = [dict(dim=2, size=n, plm='plm cons', slope_limiter='minmod', integrator=integ, cfl=.3, boundary='freeflow',
                precision='double', fast_math=True) for n in ((70, 33), (40, 51))]
    cfgs = [make_cfg(**kw) for kw in kws]
    b, alone = HipBatch(kws), HipBatch(kws[:1])
    for i, c in enumerate(cfgs):
        b.upload(i, _state(c, False))
    alone.upload(0, _state(cfgs[0], False))
    for v in (b, alone):
        v.constrainU()
        v.update(2)
    for out in (1, 2, 3):
        held = b.download(0)
        b.setActive(0, False)
        b.update(out)
        assert np.array_equal(b.download(0), held), out
        b.setActive(0, True)
        for v in (b, alone):
            v.update(2)
        assert np.array_equal(b.download(0), alone.download(0)), out
        assert b.time(0) == alone.time(0), out
