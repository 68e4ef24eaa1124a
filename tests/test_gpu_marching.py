"""The marching 2D kernel (rows per wave set) in every flux, reconstruction and math
policy, on grids where the tile kernel is the default and the other tests hold that
one to the oracle: the two advance a grid to the same bits, in finite numbers. Then
the rows a marching wave leaves to the general Roe form, on flows with many of
them, against the tile kernel, which has no such rows."""
import numpy as np
import pytest

from test_gpu_edge_cases import CASES, MODES

pytestmark = pytest.mark.gpu

FLUXES = ['hll', 'rusanov', 'euler-hllc', 'marquina']
KINDS = ['plm prim', 'plm eig', 'plm cons with flux', 'plm athena', 'ppm', 'plm eig prim', 'plm eig prim ref']
SCHEMES = {f'{f} {p}': dict(flux=f, usePLM=p, slopeLimiter='van Leer') for f in FLUXES for p in (None, 'plm cons')}
SCHEMES.update({f'{p} {lim}': dict(usePLM=p, slopeLimiter=lim) for p in KINDS for lim in ('van Leer', 'minmod', 'Koren')})
SCHEMES['entropy fix'] = dict(usePLM='plm cons', fluxArgs=dict(useEntropyFluxFix=True))
BOUNDARY = {'xmin': 'mirror', 'xmax': 'freeflow', 'ymin': 'periodic', 'ymax': 'periodic'}


def _run(kw, U0, steps, rows):
    from hydro.solver.hipfvsolver import HipFVSolver
    s = HipFVSolver(**kw)
    assert s.getLaunch()[0] == 1
    if rows:
        s.setLaunch(rows)
        assert s.getLaunch()[0] == rows
    s.resetState(U0.astype(s.dtype))
    s.update(steps)
    return s.UBufObj.toCPU(), s.t


def _same(kw, U0, steps, rows):
    ref = _run(kw, U0, steps, 0)
    assert np.isfinite(ref[0]).all() and np.isfinite(ref[1])
    for r in rows:
        got = _run(kw, U0, steps, r)
        assert np.array_equal(got[0], ref[0]) and got[1] == ref[1], r


@pytest.mark.parametrize('real,fast', [('double', False), ('double', True), ('float', True)])
@pytest.mark.parametrize('scheme', list(SCHEMES))
def test_same_bits_as_tile(scheme, real, fast):
    from hydro._cfg import make_cfg
    from hydro.init import euler as ie
    kw = dict(dim=2, gridSize=(150, 45), integrator='Runge-Kutta 2, TVD', cfl=.3, boundary=BOUNDARY, real=real, fastMath=fast,
              **SCHEMES[scheme])
    cfg = make_cfg(dim=2, size=(150, 45))
    U = ie.quadrant(cfg, ie.random_quadrant_states(np.random.default_rng(12)))
    _same(kw, ie.to_ghosted(cfg, U), 8, (3, 8, 13))
    # and with a third velocity component
    U[..., 3] = .1 * U[..., 0]
    U[..., 4] += .5 * U[..., 3] ** 2 / U[..., 0]
    _same(kw, ie.to_ghosted(cfg, U), 4, (4,))


@pytest.mark.parametrize('real,fast', [('double', False), ('double', True), ('float', True)])
@pytest.mark.parametrize('rec', [dict(usePLM='ppm'), dict(usePLM='plm cons', slopeLimiter='Koren'), dict(fluxLimiter='van Leer')],
                         ids=['ppm', 'plm', 'limited'])
@pytest.mark.parametrize('eqn', ['glm_maxwell', 'shallow_water'])
def test_other_equations_same_bits_as_tile(eqn, rec, real, fast):
    from hydro._cfg import make_cfg
    from hydro.init import euler as ie, glm_maxwell, shallow_water
    if eqn == 'shallow_water' and rec.get('usePLM') == 'ppm':
        pytest.skip('not of the shallow water equations')
    kw = dict(dim=2, gridSize=(130, 51), eqn=eqn, integrator='Runge-Kutta 3, TVD', cfl=.3, boundary=BOUNDARY, real=real,
              fastMath=fast, **rec)
    cfg = make_cfg(dim=2, size=(130, 51), eqn=eqn)
    U = glm_maxwell.gaussian_pulses(cfg, seed=2, conductivity=.3) if eqn == 'glm_maxwell' else shallow_water.humps(cfg, seed=2)
    _same(kw, ie.to_ghosted(cfg, U), 6, (3, 8, 13))


@pytest.mark.parametrize('mode', list(MODES))
@pytest.mark.parametrize('name,init,kw,steps', [c[:4] for c in CASES if c[2]['dim'] == 2], ids=[c[0] for c in CASES if c[2]['dim'] == 2])
def test_edge_branches_same_bits_as_tile(name, init, kw, steps, mode):
    from hydro._cfg import make_cfg
    from hydro.init import euler as ie
    cfg = make_cfg(dim=2, size=kw['gridSize'])
    _same(dict(kw, **MODES[mode]), ie.to_ghosted(cfg, init(cfg)), steps, (2, 7, 16))


@pytest.mark.parametrize('real', ['double', 'float'])
@pytest.mark.parametrize('scheme', ['none', 'plm prim'])
@pytest.mark.parametrize('bc', ['periodic', 'mirror', 'freeflow', 'fixed'])
def test_general_rows_at_the_faces(bc, scheme, real):
    """cold gas in the grid's corners and in its middle: irregular interfaces in the
    first and the last rows and columns, whose stencils reach over the faces ('plm cons'
    is not finite on such states, in the reference either)"""
    from hydro._cfg import make_cfg
    from hydro.init import euler as ie
    size = (135, 37)
    kw = dict(dim=2, gridSize=size, integrator='Runge-Kutta 2, TVD', cfl=.3, real=real, fastMath=True, boundary=bc,
              usePLM=None if scheme == 'none' else scheme, slopeLimiter='minmod', boundaryFixed={
                  f: [1., .1, -.1, 0., 2.5, 0.] for f in ('xmin', 'xmax', 'ymin', 'ymax')})
    cfg = make_cfg(dim=2, size=size)
    x, y, z = ie.mesh(cfg)
    thin = np.broadcast_to((np.abs(x) + np.abs(y) > 1.5) | (x * x + y * y < .05), ie.interior_shape(cfg))
    zero = np.zeros(thin.shape)
    U = ie.cons_from_prim(np.where(thin, 2e-6, 1.), (zero, zero, zero), np.where(thin, 2e-6, 1.), 1.4)
    for velocity in (False, True):
        if velocity:
            U[..., 3] = .1 * U[..., 0]
            U[..., 4] += .5 * U[..., 3] ** 2 / U[..., 0]
        _same(kw, ie.to_ghosted(cfg, U), 6, (3, 5, 16))
