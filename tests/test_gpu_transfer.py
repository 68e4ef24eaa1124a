"""Uploads and downloads of the ghosted cons_t buffer through the pinned slots
(buffers from 96 KiB on; one thread, and from some MiB on several): what comes
back is what went up, with the ghosts the oracle's boundary() fills. Every value
is copied or negated, never computed with, so the comparison is exact."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    ('1d', 1, (4099,), 'euler'), ('1d-long', 1, (200003,), 'euler'),
    ('2d', 2, (131, 77), 'euler'), ('2d-big', 2, (701, 613), 'euler'), ('2d-row', 2, (20001, 2), 'euler'),
    ('2d-column', 2, (1, 3001), 'euler'), ('3d', 3, (37, 21, 18), 'euler'), ('3d-big', 3, (70, 65, 66), 'euler'),
    ('glm', 2, (67, 53), 'glm_maxwell'), ('glm-big', 2, (301, 280), 'glm_maxwell'), ('sw', 2, (130, 63), 'shallow_water'),
    ('sw-big', 2, (512, 400), 'shallow_water'),
]


def _solver(dim, size, eqn, bc, real):
    from hydro.solver.hipfvsolver import HipFVSolver
    nstates = {'euler': 6, 'glm_maxwell': 12, 'shallow_water': 5}[eqn]
    fixed = {f: list(np.arange(1, nstates + 1) + 10. * i) for i, f in enumerate(('xmin', 'xmax', 'ymin', 'ymax', 'zmin', 'zmax'))}
    return HipFVSolver(dim=dim, gridSize=size, eqn=eqn, boundary=bc, boundaryFixed=fixed, real=real), fixed


def _ghosted(U, dim, bc, fixed, eqn):
    """U with its ghosts filled axis by axis: an index map per ghost (clamped
    to the grid where it is narrower than the ghosts), sign flips of the
    reflected fields, fixed values"""
    out = U.copy()
    faces = ('xmin', 'xmax', 'ymin', 'ymax', 'zmin', 'zmax')
    for a in range(dim):
        d = 2 - a
        n = U.shape[d] - 4
        v = np.moveaxis(out, d, 0)
        for c in (-2, -1, n, n + 1):
            side = 2 * a + (c >= n)
            kind = bc if isinstance(bc, str) else bc[faces[side]]
            src = {'periodic': c % n, 'mirror': -1 - c if c < 0 else 2 * n - 1 - c}.get(kind, 0 if c < 0 else n - 1)
            v[c + 2] = v[min(max(src, 0), n - 1) + 2]
            if kind == 'mirror':
                for f in ((a, 3 + a) if eqn == 'glm_maxwell' else (1 + a,)):
                    v[c + 2][..., f] *= -1
            if kind == 'fixed':
                v[c + 2] = np.array(fixed[faces[side]], dtype=U.dtype)
    return out


@pytest.mark.parametrize('real', ['double', 'float'])
@pytest.mark.parametrize('bc', ['periodic', 'mirror', 'freeflow', 'mixed'])
@pytest.mark.parametrize('name,dim,size,eqn', CASES, ids=[c[0] for c in CASES])
def test_round_trip(name, dim, size, eqn, bc, real):
    import pyoracle
    bc = {'xmin': 'fixed', 'xmax': 'mirror', 'ymin': 'mirror', 'ymax': 'fixed', 'zmin': 'freeflow', 'zmax': 'fixed'} \
        if bc == 'mixed' else bc
    s, fixed = _solver(dim, size, eqn, bc, real)
    assert int(np.prod(s.shape)) * s.dtype().itemsize >= 96 << 10
    rng = np.random.default_rng(3)
    U = rng.uniform(.5, 1.5, s.shape).astype(s.dtype)
    s.UBufObj.fromCPU(U)
    got = s.UBufObj.toCPU()
    assert np.array_equal(got, _ghosted(U, dim, bc, fixed, eqn))
    if min(size) < 2:     # the oracle's mirror reads a ghost there
        return
    o = pyoracle.Oracle(pyoracle.make_cfg(dim=dim, size=size, eqn=eqn, boundary=bc, boundary_fixed=fixed))
    o.set_U(U.astype(np.float64))
    o.boundary()
    assert np.array_equal(got, o.U.astype(s.dtype))


def test_out_of_plane_momentum_and_ePot():
    """what an upload finds beyond the planes: one momentum out of the plane and
    one ePot anywhere, and their absence in the next upload"""
    s, _ = _solver(2, (300, 200), 'euler', 'periodic', 'double')
    U = np.zeros(s.shape)
    U[..., 0], U[..., 4] = 1., 2.5
    for f, at in ((3, (0, 150, 7)), (5, (0, 2, 301))):
        V = U.copy()
        V[at][f] = .25
        s.UBufObj.fromCPU(V)
        s.update(1)                       # the stage kernels for three velocity components, or two
        got = s.interior(s.UBufObj.toCPU())
        assert got[..., f].max() > .1
        s.UBufObj.fromCPU(U)
        assert np.array_equal(s.interior(s.UBufObj.toCPU()), s.interior(U))


def test_threads_share_the_slots():
    """more transfers at once than there are slots for: each gets its own data"""
    bad = []

    def work(k):
        s, _ = _solver(2, (600, 401 + k), 'euler', 'periodic', 'double')
        for i in range(4):
            U = np.full(s.shape, 1. + k + 10 * i)
            s.UBufObj.fromCPU(U)
            if not np.array_equal(s.interior(s.UBufObj.toCPU())[..., :5], s.interior(U)[..., :5]):
                bad.append((k, i))
    th = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
