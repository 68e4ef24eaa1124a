"""constrainU (euler.cl:697-717) at the limits a caller may set: pressure limits
below, at and above 0, a density limit below 0, a heat capacity ratio below 1 (all
of which the reference's arithmetic takes), on states on both sides of each limit,
against the oracle. The clamps are comparisons and a handful of operations: a
field is within 16 roundings of its largest term."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIMITS = [dict(), dict(P_min=-.5), dict(P_min=.7), dict(P_min=0.), dict(rho_min=-2.), dict(rho_min=.9, P_min=-.1), dict(gamma=.8),
          dict(gamma=.8, P_min=-.2), dict(gamma=1.9, P_min=1.)]


@pytest.mark.parametrize('real,fast', [('double', True), ('float', True), ('double', False)])
@pytest.mark.parametrize('limits', LIMITS, ids=[','.join(f'{k}={v}' for k, v in d.items()) or 'default' for d in LIMITS])
def test_constrainU_limits(limits, real, fast):
    import pyoracle
    from hydro._cfg import make_cfg
    from hydro.solver.batch import HipBatch
    kw = dict(dim=2, size=(40, 30), boundary='freeflow', integrator='Runge-Kutta 2, TVD', **limits)
    b = HipBatch([dict(kw, precision=real, fast_math=fast)])
    rng = np.random.default_rng(5)
    U = np.zeros(b.shapes[0])
    sign = np.where(rng.uniform(size=U.shape[:3]) < .2, -1., 1.) if limits.get('rho_min', 0.) < 0 else 1.
    U[..., 0] = rng.uniform(.3, 1.5, U.shape[:3]) * sign
    U[..., 1:4] = rng.uniform(-1, 1, U.shape[:3] + (3,))
    U[..., 4] = rng.uniform(-2, 3, U.shape[:3])
    U = U.astype(b.dtype)
    b.upload(0, U)
    b.constrainU()
    got = b.download(0)[:, 2:-2, 2:-2, :5].astype(np.float64)
    o = pyoracle.Oracle(make_cfg(**kw))
    o.set_U(U.astype(np.float64))
    o.constrain_U()
    ref = o.U[:, 2:-2, 2:-2, :5]
    eps = 2. ** -52 if real == 'double' else 2. ** -23
    scale = np.abs(ref)
    # the energy's terms: the kinetic part, and the internal one either side of the clamp
    scale[..., 4] += np.abs(U[:, 2:-2, 2:-2, 4]) + (ref[..., 1:4] ** 2).sum(-1) / np.abs(ref[..., 0])
    assert np.all(np.abs(got - ref) <= 16 * eps * scale), np.abs((got - ref) / scale).max() / eps
