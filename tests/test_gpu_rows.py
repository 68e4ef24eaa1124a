"""GPU: the rows a wave marches, taken by the load (solver, batch, server), give
the bits of any other rows, at loads below and above one round of the device."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EQNS = ['euler', 'glm_maxwell', 'shallow_water']


def _cfg(n, eqn, real):
    return dict(dim=2, size=n, mins=(-.4, -.5), maxs=(.6, .5), eqn=eqn, plm='plm cons', slope_limiter='van Leer',
                    integrator='Runge-Kutta 2, TVD', cfl=.4, boundary='freeflow', precision=real, fast_math=True)


def _state(cfg, eqn, real):
    from hydro._cfg import make_cfg
    from hydro.init import euler as ie, glm_maxwell as ig, shallow_water as isw
    cfg = make_cfg(**cfg)
    U = ie.kelvin_helmholtz(cfg) if eqn == 'euler' else ig.gaussian_pulses(cfg) if eqn == 'glm_maxwell' else isw.humps(cfg)
    return ie.to_ghosted(cfg, U).astype('f4' if real == 'float' else 'f8')


@pytest.mark.parametrize('eqn', EQNS)
@pytest.mark.parametrize('real', ['double', 'float'])
@pytest.mark.parametrize('sizes', [[(61, 5), (64, 64), (131, 77)], [(300, 211)] * 7 + [(513, 250)] * 4])
def test_batch_and_server(eqn, real, sizes):
    from hydro.serve import Server
    from hydro.solver.batch import HipBatch
    cfgs = [_cfg(n, eqn, real) for n in sizes]
    states = [_state(c, eqn, real) for c in cfgs]
    steps, out = 4, []
    b = HipBatch(cfgs)
    rows, _ = b.getLaunch()
    assert 2 <= rows <= 32
    for r in (0, 12):
        b.setLaunch(r, 0)
        for i, U in enumerate(states):
            b.upload(i, U)
        b.update(steps)
        out.append([b.download(i) for i in range(len(b))])
    for r in (0, 12):
        s = Server(1 << 28, steps_per_tick=3)
        s.setLaunch(r, 0)
        ids = [s.submit(c, U, steps) for c, U in zip(cfgs, states)]
        done = 0
        while done < len(ids):
            s.tick()
            done = len(s.poll())
        out.append([s.result(i)[0] for i in ids])
    for got in out[1:]:
        for a, g in zip(out[0], got):
            assert np.array_equal(a, g)


@pytest.mark.parametrize('eqn', EQNS)
@pytest.mark.parametrize('real', ['double', 'float'])
@pytest.mark.parametrize('size', [(515, 491), (1100, 700)])
def test_plain(eqn, real, size):
    from hydro.solver.hipfvsolver import HipFVSolver
    out = []
    for r in (0, 3, 16):
        s = HipFVSolver(dim=2, gridSize=size, mins=(-.4, -.5), maxs=(.6, .5), eqn=eqn, usePLM='plm cons',
                        slopeLimiter='van Leer', integrator='Runge-Kutta 2, TVD', cfl=.4, boundary='freeflow', real=real,
                        fastMath=True)
        assert 2 <= s.getLaunch()[0] <= 16
        s.setLaunch(r)
        s.resetState(_state(_cfg(size, eqn, real), eqn, real))
        s.update(3)
        out.append(s.UBufObj.toCPU())
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])
