"""The 2D stage kernel's two cuts: the tile kernel (one row per wave, the
default on grids that do not fill the device) and the marching kernel (rows
per wave set) advance a grid to the same bits, whatever the scheme, type,
boundary and size. The interfaces are the same arithmetic on the same states in
both, so the comparison is exact. At these sizes it is the tile kernel that the
other tests hold to the oracle; test_gpu_marching compares the marching kernel of
the schemes not listed here."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# sizes at the edges of a tile (3 rows; 60 or 64 columns) and of a block row
SIZES = [(1, 1), (3, 2), (59, 3), (60, 4), (61, 7), (64, 6), (65, 1), (130, 11)]
SCHEMES = {
    'plm': dict(usePLM='plm cons'),
    'plm-vl': dict(usePLM='plm cons', slopeLimiter='van Leer'),
    'plm-rt': dict(usePLM='plm cons', slopeLimiter='Koren'),
    'superbee': dict(fluxLimiter='superbee'),
    'van-leer': dict(fluxLimiter='van Leer', integrator='Runge-Kutta 3, TVD'),
    'donor': dict(),
    'rk4': dict(usePLM='plm cons', integrator='Runge-Kutta 4'),
    'hllc': dict(usePLM='plm cons', flux='euler-hllc'),
    'eig': dict(usePLM='plm eig'),
    'athena': dict(usePLM='plm athena'),
    'fix': dict(fluxLimiter='superbee', fluxArgs=dict(useEntropyFluxFix=True)),
    'fixed-dt': dict(usePLM='plm cons', fixedDT=1e-3),
}
EULER_ONLY = ('hllc', 'eig', 'athena', 'fix')


def _initial(eqn, cfg):
    from hydro.init import euler, glm_maxwell, shallow_water
    if eqn == 'glm_maxwell':
        return glm_maxwell.gaussian_pulses(cfg, seed=2, conductivity=.3)
    if eqn == 'shallow_water':
        return shallow_water.humps(cfg, seed=2)
    rng = np.random.default_rng(2)
    U = euler.quadrant(cfg, euler.random_quadrant_states(rng))
    # an out-of-plane momentum: three velocity components
    U[..., 3] = .1 * U[..., 0]
    U[..., 4] += .5 * U[..., 3] ** 2 / U[..., 0]
    return U


@pytest.mark.parametrize('eqn', ['euler', 'glm_maxwell', 'shallow_water'])
@pytest.mark.parametrize('scheme', list(SCHEMES))
@pytest.mark.parametrize('real,fast', [('double', True), ('float', True), ('double', False)])
def test_tile_same_bits_as_marching(eqn, scheme, real, fast):
    from hydro.init import euler as init_euler
    from hydro.solver.hipfvsolver import HipFVSolver
    if eqn != 'euler' and scheme in EULER_ONLY:
        pytest.skip('an Euler scheme')
    kw = dict(dict(dim=2, eqn=eqn, integrator='Runge-Kutta 2, TVD', cfl=.3, real=real, fastMath=fast), **SCHEMES[scheme])
    for i, size in enumerate(SIZES):
        bc = ('periodic', 'mirror', 'freeflow')[i % 3]
        if eqn == 'euler' and i % 4 == 3:
            bc = {'xmin': 'fixed', 'ymax': 'fixed'}
            kw['boundaryFixed'] = {'xmin': [1., .3, 0., .1, 3., 0.], 'ymax': [.5, 0., -.1, 0., 1., 0.]}
        s = HipFVSolver(gridSize=size, boundary=bc, **kw)
        assert s.getLaunch()[0] == 1
        U0 = init_euler.to_ghosted(s.cfg, _initial(eqn, s.cfg)).astype(s.dtype)
        m = HipFVSolver(gridSize=size, boundary=bc, **kw)
        m.setLaunch(4)
        for v in (s, m):
            v.resetState(U0)
            v.update(6)
        assert np.array_equal(s.UBufObj.toCPU(), m.UBufObj.toCPU(), equal_nan=True), (size, bc)
        assert s.t == m.t, (size, bc)


def test_tile_general_form():
    """Vacuum next to gas: the tile kernel's interfaces of the general Roe form
    against the marching kernel's rows of it"""
    from hydro.init import euler as init_euler
    from hydro.solver.hipfvsolver import HipFVSolver
    for real in ('double', 'float'):
        kw = dict(dim=2, gridSize=(130, 17), usePLM='plm cons', integrator='Runge-Kutta 2, TVD', cfl=.3, real=real,
                  boundary='freeflow', fastMath=True, eqnArgs=dict(rhoMin=1e-7))
        out = []
        for rows in (0, 4, 16):
            s = HipFVSolver(**kw)
            if rows:
                s.setLaunch(rows)
            U = init_euler.riemann(s.cfg, {'rho': 1., 'P': 1., 'v': (.2, -.3, 0.)}, {'rho': 1e-6, 'P': 1e-6}, 1.4)
            s.resetState(init_euler.to_ghosted(s.cfg, U).astype(s.dtype))
            s.update(15)
            out.append((s.UBufObj.toCPU(), s.t))
        for U, t in out[1:]:
            assert np.array_equal(U, out[0][0]) and t == out[0][1]
