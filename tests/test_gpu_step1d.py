"""Whole 1D integrator steps per launch (several of them where the grid fits one
block) against one launch per stage, which the batched form takes: the same
arithmetic on the same states, so the same bits, in every scheme, integrator,
type and boundary, at sizes around the waves' 60 .. 48 output cells, the one-block
limit and below the halo's width."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 5, 48, 61, 113, 383, 449, 481, 1000]
SCHEMES = {
    'fe-superbee': dict(flux_limiter='superbee', integrator='forward Euler'),
    'rk2-plm': dict(plm='plm cons', integrator='Runge-Kutta 2, TVD'),
    'rk2-heun-vl': dict(flux_limiter='van Leer', integrator='Runge-Kutta 2 Heun'),
    'rk3-donor': dict(integrator='Runge-Kutta 3, TVD'),
    'rk4-plm': dict(plm='plm cons', slope_limiter='Koren', integrator='Runge-Kutta 4'),
    'rk4-tvd': dict(plm='plm cons', slope_limiter='superbee', integrator='Runge-Kutta 4, TVD'),
    'fixed-dt': dict(plm='plm cons', integrator='Runge-Kutta 3', fixed_dt=2e-4),
    'hll': dict(flux='hll', plm='plm cons', integrator='Runge-Kutta 2, TVD'),
    'eig': dict(plm='plm eig', integrator='Runge-Kutta 2, TVD'),
}
BCS = ['periodic', 'freeflow', 'mirror', {'xmin': 'fixed', 'xmax': 'mirror'}, {'xmin': 'periodic', 'xmax': 'freeflow'}]
FIXED = {'xmin': [1., .2, .1, 0., 2.5, 0.]}


def _initial(cfg, eqn, n):
    from hydro.init import euler, glm_maxwell, shallow_water
    if eqn == 'glm_maxwell':
        return glm_maxwell.gaussian_pulses(cfg, seed=4, conductivity=.2)
    if eqn == 'shallow_water':
        return shallow_water.humps(cfg, seed=4)
    rng = np.random.default_rng(n)
    U = euler.riemann(cfg, {'rho': 1.2, 'P': 1., 'v': (.3, .2, 0.)}, {'rho': .3, 'P': .2, 'v': (-.1, 0., .1)}, 1.4)
    U[..., 0] *= 1 + .05 * rng.uniform(-1, 1, U.shape[:-1])
    return U


@pytest.mark.parametrize('real,fast', [('double', True), ('float', True), ('double', False)])
@pytest.mark.parametrize('scheme', list(SCHEMES))
@pytest.mark.parametrize('eqn', ['euler', 'glm_maxwell', 'shallow_water'])
def test_same_bits_as_batched_stages(eqn, scheme, real, fast):
    from hydro._cfg import make_cfg
    from hydro.init import euler as init_euler
    from hydro.solver.batch import HipBatch
    from hydro.solver.hipfvsolver import HipFVSolver
    if eqn != 'euler' and scheme in ('hll', 'eig'):
        pytest.skip('an Euler scheme')
    for i, n in enumerate(SIZES):
        bc = BCS[i % len(BCS)] if eqn == 'euler' else BCS[i % 3]
        kw = dict(dict(dim=1, size=n, eqn=eqn, boundary=bc, boundary_fixed=FIXED, cfl=.3, precision=real, fast_math=fast),
                  **SCHEMES[scheme])
        cfg = make_cfg(**kw)
        U = init_euler.to_ghosted(cfg, _initial(cfg, eqn, n))
        b = HipBatch([kw])
        s = HipFVSolver(dim=1, gridSize=(n,), eqn=eqn, boundary=bc, boundaryFixed=FIXED, cfl=.3, real=real, fastMath=fast,
                        usePLM=kw.get('plm'), slopeLimiter=kw.get('slope_limiter', 'minmod'), flux=kw.get('flux', 'roe'),
                        fluxLimiter=kw.get('flux_limiter', 'donor cell'), integrator=kw['integrator'],
                        fixedDT=kw.get('fixed_dt'))
        U = U.astype(s.dtype)
        b.upload(0, U)
        b.constrainU()
        s.resetState(U)
        for steps in (1, 7, 300 if n in (48, 383) else 2):
            b.update(steps, graph=False)
            s.update(steps)
            assert np.array_equal(s.UBufObj.toCPU(), b.download(0), equal_nan=True), (n, bc, steps)
            assert (s.t, s.dt) == b.time(0), (n, bc, steps)
        # a step of the caller's, then steps of its own again
        if 'fixed_dt' not in kw:
            dt = s.calcDT()
            assert dt > 0
            s.step(.5 * dt)
            s.update(3)
            assert np.isfinite(s.UBufObj.toCPU()).all()
