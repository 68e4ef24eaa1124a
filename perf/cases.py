"""The work a user of this framework has it do, as cases that can be timed and
compared: solves, snapshots of a running simulation, a live view, an ensemble
advanced together and a stream of served requests, through the public classes
(HipFVSolver, HipBatch, Server).

Kinds of pass (`kind`):
  solve     a new initial state goes up, `steps` updates, the final state comes
            down: one problem of a parameter study or a convergence test
  snapshot  a running simulation advances `steps` updates and its state comes
            down for a dump or a plot
  live      `steps` frames of one update each, with the time and the display
            range and statistics of two variables read after every frame, as
            the reference's interactive view does; then one download
  batch     an ensemble of uneven grids: all states up, `steps` updates
            together, all states down
  serve     a set of solve requests through the server: submitted at once,
            ticked until done, every result fetched

exact() is an independent finite-volume solver in float64 on torch tensors.
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'hydro-cl-lua_amd'))

GAMMA = 1.4
RHO_MIN = P_MIN = 1e-7
NG = 2
DEV = 'cuda' if torch.cuda.is_available() else 'cpu'

FE, RK2, RK3 = 'forward Euler', 'Runge-Kutta 2, TVD', 'Runge-Kutta 3, TVD'

# Largest box of a batch or served request that exact() computes, and how many.
EXACT_CELLS, EXACT_GRIDS = 160 * 160, 4


def plain(name, kind, nx, ny, nz, steps, init, **kw):
    """a case of one grid; ny = nz = 1 for 1D, nz = 1 for 2D"""
    c = dict(kind=kind, nx=nx, ny=ny, nz=nz, steps=steps, init=init, eqn='euler', real='double', fast=True,
             plm='plm cons', limiter='minmod', integrator=RK2, cfl=.4, boundary='periodic')
    c.update(kw)
    if name:
        c['name'] = name
    return c


def listed():
    return [
        # the smallest: Sod's tube on 256 cells, the reference's first example,
        # in its own arithmetic (IEEE) with its default scheme (Roe with a flux
        # limiter, forward Euler): launches and transfers are all there is
        plain('sod_256', 'solve', 256, 1, 1, 100, 'sod', fast=False, plm='', limiter='superbee', integrator=FE, cfl=.5,
              boundary='fixed'),
        # a long 1D Riemann problem at an odd length, the 1D requests of the
        # serving mix run alone
        plain('riemann_20011_f32', 'solve', 20011, 1, 1, 400, 'riemann', real='float', boundary='freeflow'),
        # the reference's default view: 256^2, Roe with superbee, forward Euler,
        # one update per frame with the displayed ranges
        plain('live_256', 'live', 256, 256, 1, 20, 'kh', plm='', limiter='superbee', integrator=FE, cfl=.5),
        # the headline: Kelvin-Helmholtz 1024^2 FP64, RK2-TVD, 500 steps
        plain('kh_1024', 'snapshot', 1024, 1024, 1, 500, 'kh'),
        # the same flow beyond the last-level cache (U^n and U^1 are 336 MB)
        plain('kh_2048', 'snapshot', 2048, 2048, 1, 300, 'kh'),
        # FP32 on an odd, ragged grid with open edges, another slope limiter
        # and the third-order integrator
        plain('quadrants_1501x997_f32', 'solve', 1501, 997, 1, 200, 'quadrants', real='float', limiter='van Leer',
              integrator=RK3, boundary='freeflow'),
        # the constructor's default arithmetic (IEEE division and square root),
        # between mirror walls
        plain('kh_600x400_ieee', 'snapshot', 600, 400, 1, 200, 'kh', fast=False, boundary='mirror'),
        # 3D: the spherical blast at its full size, FP32, van Leer flux
        # limiter, RK3-TVD
        plain('blast_256_f32', 'snapshot', 256, 256, 256, 100, 'blast', real='float', plm='', limiter='van Leer',
              integrator=RK3, cfl=.3, boundary='freeflow'),
        # the other equations: Maxwell with cleaning fields, conducting medium
        plain('maxwell_512_f32', 'solve', 512, 512, 1, 400, 'pulses', eqn='glm_maxwell', real='float'),
        # ... and shallow water over a bumpy bottom
        plain('lake_700x500', 'solve', 700, 500, 1, 300, 'humps', eqn='shallow_water', boundary='freeflow'),
        # an ensemble of uneven four-quadrant problems, sides 64..512
        dict(name='ensemble_48_f32', kind='batch', count=48, lo=64, hi=512, steps=200, real='float', mix=1),
        # served requests: 1D Euler, 2D Euler and 2D Maxwell, mixed
        dict(name='serve_24_f32', kind='serve', count=24, lo=64, hi=768, steps=300, real='float', mix=2),
    ]


def draw(rng):
    """One more case: sizes log-uniform and mostly odd, options as in listed()."""
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    real, bc = rng.choice(['double', 'float']), rng.choice(['periodic', 'freeflow', 'mirror'])
    pick = rng.randrange(8)
    if pick == 0:
        return dict(kind='batch', count=logint(6, 56), lo=logint(48, 96), hi=logint(200, 480), steps=logint(50, 200),
                    real=real, mix=rng.randrange(1 << 20))
    if pick == 1:
        return dict(kind='serve', count=logint(4, 24), lo=logint(48, 96), hi=logint(200, 640), steps=logint(50, 300),
                    real=real, mix=rng.randrange(1 << 20))
    limited = rng.random() < .4      # flux limiter instead of a reconstruction
    kw = dict(real=real, fast=rng.random() < .8, boundary=bc, plm='' if limited else 'plm cons',
              limiter=rng.choice(['minmod', 'superbee', 'van Leer']), integrator=rng.choice([FE, RK2, RK2, RK3]))
    if kw['integrator'] == FE and not limited:
        kw['integrator'] = RK2       # a reconstruction without a Runge-Kutta integrator is not stable
    if pick == 2:
        return plain('', 'solve', logint(256, 65536), 1, 1, logint(50, 500), 'riemann', **dict(kw, boundary='freeflow'))
    if pick == 3:
        return plain('', 'live', logint(48, 500), logint(48, 500), 1, logint(8, 30), 'kh', **dict(kw, fast=True))
    if pick == 4:
        return plain('', 'snapshot', logint(60, 200), logint(60, 200), logint(60, 200), logint(10, 40), 'blast',
                     **dict(kw, cfl=.3, boundary='freeflow'))
    if pick == 5:
        if rng.random() < .5:
            return plain('', 'solve', logint(64, 900), logint(64, 900), 1, logint(50, 200), 'pulses', eqn='glm_maxwell',
                         real=real, limiter=kw['limiter'])
        return plain('', 'solve', logint(64, 1200), logint(64, 1200), 1, logint(50, 200), 'humps', eqn='shallow_water',
                     real=real, limiter=kw['limiter'], boundary='freeflow')
    return plain('', rng.choice(['solve', 'snapshot']), logint(64, 2000), logint(64, 2000), 1, logint(50, 200),
                 'kh' if bc != 'freeflow' else 'quadrants', **kw)


# ------------------------------------------------------------ initial states
# Interior cons_t fields as one float64 tensor (S, z, y, x).

def box(case):
    """the domain: cells of about 1/1000 at the 2D sizes (the reference takes a
    cell below 1e-7 in volume as solid), [-1, 1] in 1D and 3D"""
    dim = dim_of(case)
    if dim != 2:
        return (-1.,) * dim, (1.,) * dim
    s = max(1., case['nx'] / 1024., case['ny'] / 1024.)
    return (-.5 * s, -.5 * s), (.5 * s, .5 * s)


def dim_of(case):
    return 1 if case['ny'] == 1 and case['nz'] == 1 else 2 if case['nz'] == 1 else 3


def coords(case):
    dim = dim_of(case)
    lo, hi = box(case)
    n = (case['nx'], case['ny'], case['nz'])
    out = []
    for i in range(3):
        if i < dim:
            c = (torch.arange(n[i], dtype=torch.float64, device=DEV) + .5) / n[i] * (hi[i] - lo[i]) + lo[i]
        else:
            c = torch.zeros(1, dtype=torch.float64, device=DEV)
        out.append(c.view([-1 if k == 2 - i else 1 for k in range(3)]))
    return out


def euler_cons(rho, v, P, shape):
    full = [torch.as_tensor(a, dtype=torch.float64, device=DEV).expand(shape) for a in (rho, *v, P)]
    rho, vx, vy, vz, P = full
    E = .5 * rho * (vx * vx + vy * vy + vz * vz) + P / (GAMMA - 1)
    return torch.stack([rho, rho * vx, rho * vy, rho * vz, E, torch.zeros_like(rho)])


SOD = ((1., 1.), (.125, .1))        # (rho, P) of the two sides


def initial(case, seed):
    x, y, z = coords(case)
    shape = (case['nz'], case['ny'], case['nx'])
    rng = random.Random(seed * 7919 + 13)
    lo, hi = box(case)
    kind = case['init']
    if kind == 'sod':
        # the tube with its two states scaled by a per cent or so
        f = [1 + rng.uniform(-.02, .02) for _ in range(4)]
        left = x < 0
        rho = torch.where(left, SOD[0][0] * f[0], SOD[1][0] * f[1])
        P = torch.where(left, SOD[0][1] * f[2], SOD[1][1] * f[3])
        return euler_cons(rho, (0., 0., 0.), P, shape)
    if kind == 'riemann':
        s = [(rng.uniform(.1, 2), rng.uniform(-.5, .5), rng.uniform(.1, 2)) for _ in range(2)]
        left = x < 0
        rho, vx, P = (torch.where(left, s[0][k], s[1][k]) for k in range(3))
        return euler_cons(rho, (vx, 0., 0.), P, shape)
    if kind == 'kh':
        gen = torch.Generator(device=DEV).manual_seed(seed)
        h = hi[1] - lo[1]
        inside = (y - .5 * (lo[1] + hi[1])).abs() < .25 * h
        noise = (torch.rand(shape, generator=gen, dtype=torch.float64, device=DEV) * 2 - 1) * 1e-3
        theta = 4 * math.pi * (x - lo[0]) / (hi[0] - lo[0]) + rng.uniform(0, 2 * math.pi)
        vy = .01 * torch.sin(theta) + noise
        return euler_cons(torch.where(inside, 2., 1.), (torch.where(inside, .5, -.5), vy, 0.), 2.5, shape)
    if kind == 'quadrants':
        s = []
        for _ in range(4):
            r, t = rng.uniform(0, .5), rng.uniform(0, 2 * math.pi)
            s.append((rng.uniform(.1, 2), r * math.cos(t), r * math.sin(t), rng.uniform(.1, 2)))
        right, top = (x > .5 * (lo[0] + hi[0])), (y > .5 * (lo[1] + hi[1]))
        rho, vx, vy, P = (torch.where(top, torch.where(right, s[0][k], s[1][k]), torch.where(right, s[3][k], s[2][k]))
                          for k in range(4))
        return euler_cons(rho, (vx, vy, 0.), P, shape)
    if kind == 'blast':
        c = [rng.uniform(lo[i] + .25 * (hi[i] - lo[i]), hi[i] - .25 * (hi[i] - lo[i])) for i in range(3)]
        r2 = (x - c[0]) ** 2 + (y - c[1]) ** 2 + (z - c[2]) ** 2
        return euler_cons(1., (0., 0., 0.), torch.where(r2 < .01, 10., .1), shape)
    # Gaussian bumps, for the other two equations
    bumps = []
    for _ in range(3):
        c = [rng.uniform(lo[i] + .3 * (hi[i] - lo[i]), hi[i] - .3 * (hi[i] - lo[i])) for i in range(2)]
        w = rng.uniform(.05, .15) * (hi[0] - lo[0])
        bumps.append(torch.exp(-((x - c[0]) ** 2 + (y - c[1]) ** 2) / (w * w)))
    if kind == 'pulses':
        U = torch.zeros((12,) + shape, dtype=torch.float64, device=DEV)
        for b in bumps[:2]:
            for k in range(6):
                U[k] += rng.uniform(-1, 1) * b
        U[9] = .5 * bumps[2]            # conductivity
        U[10] = U[11] = 1.              # sqrt(1 / eps), sqrt(1 / mu)
        return U
    U = torch.zeros((5,) + shape, dtype=torch.float64, device=DEV)
    U[0] = 1.
    U[4] = .2 * rng.uniform(-1, 1) * x + .2 * rng.uniform(-1, 1) * y
    for b in bumps:
        U[0] += rng.uniform(.1, .3) * b
        U[4] += .1 * rng.uniform(-1, 1) * b
        U[1] += .2 * rng.uniform(-1, 1) * b
        U[2] += .2 * rng.uniform(-1, 1) * b
    U[1:3] *= U[0]
    return U


def dtype_of(case):
    return np.float64 if case['real'] == 'double' else np.float32


def host_state(case, U):
    """the ghosted cons_t buffer (z, y, x, S) a user has in hand (ghosts zero)"""
    dim = dim_of(case)
    g = [s + (2 * NG if i < dim else 0) for i, s in enumerate((case['nx'], case['ny'], case['nz']))]
    out = np.zeros((g[2], g[1], g[0], U.shape[0]), dtype=dtype_of(case))
    sl = tuple(slice(NG, -NG) if 2 - k < dim else slice(None) for k in range(3))
    t = torch.float64 if case['real'] == 'double' else torch.float32
    out[sl] = U.permute(1, 2, 3, 0).to(t).cpu().numpy()
    return out


def fixed_values(case, U):
    """the ghost values of a tube held at its two end states"""
    return {'xmin': U[:, 0, 0, 0].tolist(), 'xmax': U[:, 0, 0, -1].tolist()}


def arguments(case):
    """HipFVSolver's arguments for a case of one grid"""
    dim = dim_of(case)
    lo, hi = box(case)
    lim = case['limiter']
    return dict(dim=dim, gridSize=(case['nx'], case['ny'], case['nz'])[:dim], mins=lo, maxs=hi, eqn=case['eqn'],
                flux='roe', usePLM=case['plm'] or None, slopeLimiter=lim if case['plm'] else 'minmod',
                fluxLimiter='donor cell' if case['plm'] else lim, integrator=case['integrator'], cfl=case['cfl'],
                boundary=case['boundary'], real=case['real'], fastMath=case['fast'])


def configuration(case):
    """the same as make_cfg's arguments (batch and server)"""
    a = arguments(case)
    return dict(dim=a['dim'], size=a['gridSize'], mins=a['mins'], maxs=a['maxs'], eqn=a['eqn'], plm=a['usePLM'],
                slope_limiter=a['slopeLimiter'], flux_limiter=a['fluxLimiter'], integrator=a['integrator'],
                cfl=a['cfl'], boundary=a['boundary'], precision=a['real'], fast_math=a['fastMath'])


def members(case):
    """the grids of a batch or the requests of a served set: plain cases. The
    shapes and step counts come from the case (`mix`), the states from the
    seed."""
    rng = random.Random(case['mix'])
    out = []
    for _ in range(case['count']):
        side = [int(round(math.exp(rng.uniform(math.log(case['lo']), math.log(case['hi']))))) for _ in range(2)]
        if case['kind'] == 'batch':
            out.append(plain('', 'solve', side[0], side[0], 1, case['steps'], 'quadrants', real=case['real'],
                             boundary='freeflow'))
            continue
        steps = rng.randint(max(1, case['steps'] // 10), case['steps'])
        what = rng.randrange(3)
        if what == 0:
            out.append(plain('', 'solve', rng.randint(256, 65536), 1, 1, steps, 'riemann', real=case['real'],
                             boundary='freeflow'))
        elif what == 1:
            out.append(plain('', 'solve', side[0], side[0], 1, steps, 'quadrants', real=case['real'],
                             boundary='freeflow'))
        else:
            s = max(64, side[0] * 2 // 3)
            out.append(plain('', 'solve', s, s, 1, steps, 'pulses', eqn='glm_maxwell', real=case['real']))
    return out


# ------------------------------------------------------------ the measured path

def prepare(case, seed):
    from hydro.serve import Server
    from hydro.solver.batch import HipBatch
    from hydro.solver.hipfvsolver import HipFVSolver
    if case['kind'] in ('batch', 'serve'):
        ms = members(case)
        states = [host_state(m, initial(m, seed * 1009 + i)) for i, m in enumerate(ms)]
        cfgs = [configuration(m) for m in ms]
        if case['kind'] == 'serve':
            return dict(case=case, server=Server(2 << 30, steps_per_tick=20), cfgs=cfgs, states=states,
                        steps=[m['steps'] for m in ms])
        b = HipBatch(cfgs)
        for i, U in enumerate(states):
            b.upload(i, U)
        b.constrainU()
        b.autotune(3)
        return dict(case=case, batch=b, states=states)
    U = initial(case, seed)
    args = arguments(case)
    if case['boundary'] == 'fixed':
        args['boundary'] = {'xmin': 'fixed', 'xmax': 'fixed'}
        args['boundaryFixed'] = fixed_values(case, U)
    s = HipFVSolver(**args)
    state = host_state(case, U)
    s.resetState(state)
    return dict(case=case, solver=s, state=state)


def run(state):
    case = state['case']
    kind = case['kind']
    if kind == 'batch':
        b = state['batch']
        for i, U in enumerate(state['states']):
            b.upload(i, U)
        b.constrainU()
        b.update(case['steps'])
        return [b.download(i) for i in range(len(b))]
    if kind == 'serve':
        srv = state['server']
        ids = {srv.submit(c, U, n): i for i, (c, U, n) in enumerate(zip(state['cfgs'], state['states'], state['steps']))}
        out = [None] * len(ids)
        t, status = np.zeros(len(ids)), np.zeros(len(ids), dtype=np.int64)
        while ids:
            srv.tick()
            for rid in srv.poll():
                i = ids.pop(rid)
                out[i], t[i], status[i] = srv.result(rid)
        return {'U': out, 't': t, 'status': status}
    s = state['solver']
    if kind == 'live':
        seen, times = np.zeros((case['steps'], 2, 4)), np.zeros(case['steps'])
        for k in range(case['steps']):
            s.update()
            times[k] = s.t
            seen[k, 0] = s.calcDisplayVarRangeAndAvgAndStdDev(0)
            seen[k, 1] = s.calcDisplayVarRangeAndAvgAndStdDev('P')
        return {'U': s.UBufObj.toCPU(), 'stats': seen, 't': times}
    if kind == 'solve':
        s.resetState(state['state'])
    s.update(case['steps'])
    return {'U': s.UBufObj.toCPU(), 't': s.t}


def work(case):
    """Per step and cell the state is read once and written once (and the
    static fields read once), whatever the number of stages; a pass also writes
    the ghosted cons_t buffer (and reads one when a state goes up). Flops: what
    one stage of one cell takes (two edges, one Roe flux and its share of the
    update per axis), times the stages."""
    cases = members(case) if case['kind'] in ('batch', 'serve') else [case]
    nbytes = flops = 0.
    for c in cases:
        dim, cells = dim_of(c), c['nx'] * c['ny'] * c['nz']
        w = 8 if c['real'] == 'double' else 4
        q, stat, S, per_axis = {'euler': (5, 0, 6, 150), 'glm_maxwell': (8, 4, 12, 110),
                                'shallow_water': (4, 1, 5, 110)}[c['eqn']]
        if c['eqn'] == 'euler' and dim < 3:
            q = 3 if dim == 1 else 4          # momenta out of the plane are 0
        stages = {FE: 1, RK2: 2, RK3: 3}[c['integrator']]
        nbytes += c['steps'] * cells * (2 * q + stat) * w + cells * S * w * (1 if c['kind'] == 'snapshot' else 2)
        flops += c['steps'] * stages * cells * (per_axis * dim + 40)
        if c['kind'] == 'live':
            nbytes += c['steps'] * cells * (q + 1) * w
    return {'bytes': nbytes, 'flops': flops}


# ------------------------------------------------------------ float64 reference
# Fields are tensors (q, z, y, x). Every function is written from the scheme's
# definition: MUSCL edges or a flux-limited Roe flux, unsplit divergence,
# Shu-Osher Runge-Kutta steps, CFL step from the fastest wave of any cell.

def dx_of(case):
    lo, hi = box(case)
    n = (case['nx'], case['ny'], case['nz'])
    return [(hi[i] - lo[i]) / n[i] for i in range(dim_of(case))]


def flips(case, axis):
    return (axis, 3 + axis) if case['eqn'] == 'glm_maxwell' else (1 + axis,)


def padded(case, U, axis, fixed):
    """U with two ghost layers along axis (0 x, 1 y, 2 z)"""
    d = 3 - axis
    n = U.shape[d]
    bc = case['boundary']

    def take(idx):
        return U.index_select(d, torch.tensor(idx, device=U.device))

    if bc == 'periodic':
        lo, hi = take([(-2) % n, (-1) % n]), take([0 % n, 1 % n])
    elif bc == 'mirror':
        lo, hi = take([min(1, n - 1), 0]), take([n - 1, max(n - 2, 0)])
        for f in flips(case, axis):
            lo[f], hi[f] = -lo[f], -hi[f]
    else:
        lo, hi = take([0, 0]), take([n - 1, n - 1])
        if bc == 'fixed':
            for side, g in (('xmin', lo), ('xmax', hi)):
                g[:] = fixed[side][:U.shape[0]].view(-1, 1, 1, 1)
    return torch.cat([lo, U, hi], d)


def cut(U, axis, a, b):
    return U.narrow(3 - axis, a, U.shape[3 - axis] - a - b)


def phi_times(lim, num, den):
    """phi(num / den) * den"""
    if lim == 'minmod':
        return torch.where(num * den > 0, torch.where(num.abs() < den.abs(), num, den), 0.)
    r = num / torch.where(den == 0, 1., den)
    if lim == 'superbee':
        phi = torch.clamp(torch.maximum(torch.clamp(2 * r, max=1), torch.clamp(r, max=2)), min=0)
    else:
        phi = torch.where(r > 0, 2 * r / (1 + r.clamp(min=0)), 0.)
    return torch.where(den == 0, 0., phi * den)


def prims(U):
    v = U[1:4] / U[0]
    P = (GAMMA - 1) * (U[4] - .5 * U[0] * (v * v).sum(0))
    return v, P


def euler_flux(U, v, P, a):
    F = U[:5] * v[a]
    F[1 + a] += P
    F[4] += P * v[a]
    return F


def euler_roe(L, R, a):
    """Roe state (v, H, c), characteristic jumps (wave strengths) and mean flux"""
    vL, PL = prims(L)
    vR, PR = prims(R)
    F = .5 * (euler_flux(L, vL, PL, a) + euler_flux(R, vR, PR, a))
    sL, sR = L[0].sqrt(), R[0].sqrt()
    w = sL / (sL + sR)
    v = w * vL + (1 - w) * vR
    H = w * (L[4] + PL) / L[0] + (1 - w) * (R[4] + PR) / R[0]
    q2 = .5 * (v * v).sum(0)
    c = ((GAMMA - 1) * (H - q2)).sqrt()
    d = R[:5] - L[:5]
    dp = (GAMMA - 1) * (d[4] - (v * d[1:4]).sum(0) + q2 * d[0])
    b, e = 1 + (a + 1) % 3, 1 + (a + 2) % 3
    dm = c * (v[a] * d[0] - d[1 + a])
    y = torch.stack([(dp + dm) / (2 * c * c), d[0] - dp / (c * c), d[b] - v[b - 1] * d[0], d[e] - v[e - 1] * d[0],
                     (dp - dm) / (2 * c * c)])
    lam = torch.stack([v[a] - c, v[a], v[a], v[a], v[a] + c])
    return (v, H, q2, c), y, lam, F


def euler_right(state, z, a):
    v, H, q2, c = state
    b, e = 1 + (a + 1) % 3, 1 + (a + 2) % 3
    s, t = z[0] + z[1] + z[4], z[4] - z[0]
    out = torch.empty_like(z)
    out[0] = s
    out[1 + a] = v[a] * s + c * t
    out[b] = v[b - 1] * s + z[2]
    out[e] = v[e - 1] * s + z[3]
    out[4] = H * (z[0] + z[4]) + c * v[a] * t + q2 * z[1] + v[b - 1] * z[2] + v[e - 1] * z[3]
    return out


def maxwell_flux(U, a):
    # uniform medium with eps = mu = 1 and cleaning speeds 1: every wave has speed 1
    b, e = (a + 1) % 3, (a + 2) % 3
    F = torch.zeros_like(U[:8])
    F[a], F[b], F[e] = U[6], U[3 + e], -U[3 + b]
    F[3 + a], F[3 + b], F[3 + e] = U[7], -U[e], U[b]
    F[6], F[7] = U[a], U[3 + a]
    return F


def water_flux(U, a):
    F = U[:4] * (U[1 + a] / U[0])
    F[1 + a] += .5 * U[0] * U[0]
    return F


def interface_flux(case, L, R, a):
    if case['eqn'] == 'euler':
        s, y, lam, F = euler_roe(L, R, a)
        return F - .5 * euler_right(s, lam.abs() * y, a)
    if case['eqn'] == 'glm_maxwell':
        return .5 * (maxwell_flux(L, a) + maxwell_flux(R, a)) - .5 * (R[:8] - L[:8])
    # shallow water, gravity 1: arithmetic mean height, sqrt(h)-weighted velocity
    sL, sR = L[0].sqrt(), R[0].sqrt()
    v = (L[1:4] / L[0] * sL + R[1:4] / R[0] * sR) / (sL + sR)
    h = .5 * (L[0] + R[0])
    c = h.sqrt()
    d = R[:4] - L[:4]
    vn = v[a]
    m = d[1 + a] - vn * d[0]
    am, ap = .5 * (d[0] - m / c), .5 * (d[0] + m / c)
    z0, z3, an = (vn - c).abs() * am, (vn + c).abs() * ap, vn.abs()
    D = torch.empty_like(d)
    D[0] = z0 + z3
    D[1:4] = v * (z0 + z3) + an * (d[1:4] - v * d[0])
    D[1 + a] = (vn - c) * z0 + (vn + c) * z3
    return .5 * (water_flux(L, a) + water_flux(R, a)) - .5 * D


def derivative(case, U, stat, dt, fixed):
    """-div F plus the source"""
    lim = case['limiter']
    q = U.shape[0]
    out = torch.zeros_like(U)
    for a, dx in enumerate(dx_of(case)):
        P = padded(case, U, a, fixed)
        if case['plm']:
            lo, mid, hi = cut(P, a, 0, 2), cut(P, a, 1, 1), cut(P, a, 2, 0)
            s = .5 * phi_times(lim, mid - lo, hi - mid)
            F = interface_flux(case, cut(mid + s, a, 0, 1), cut(mid - s, a, 1, 0), a)
        else:
            s, y, lam, F = euler_roe(cut(P, a, 0, 1), cut(P, a, 1, 0), a)
            y0, l0 = cut(y, a, 1, 1), cut(lam, a, 1, 1)
            up = torch.where(l0 >= 0, cut(y, a, 0, 2), cut(y, a, 2, 0))
            sgn = torch.where(l0 >= 0, 1., -1.)
            z = -.5 * l0 * (sgn * y0 + phi_times(lim, up, y0) * (l0 * dt / dx - sgn))
            s = tuple(cut(x if x.dim() == 4 else x[None], a, 1, 1) for x in s)
            s = (s[0], s[1][0], s[2][0], s[3][0])
            F = cut(F, a, 1, 1) + euler_right(s, z, a)
        out -= (cut(F, a, 1, 0) - cut(F, a, 0, 1)) / dx
        if case['eqn'] == 'shallow_water':
            D = padded(case, stat, a, fixed)      # the bottom; open or periodic edges
            out[1 + a] += U[0] * (cut(D, a, 3, 1) - cut(D, a, 1, 3))[0] / (2 * dx)
    if case['eqn'] == 'glm_maxwell':
        out[:3] -= U[:3] * stat[1]        # conductivity (eps = 1)
        out[6] += stat[0]                 # charge
    return out


def constrained(case, U):
    if case['eqn'] != 'euler':
        return U
    U = U.clone()
    U[0] = U[0].clamp(min=RHO_MIN)
    v, P = prims(U)
    U[4] = .5 * U[0] * (v * v).sum(0) + P.clamp(min=P_MIN) / (GAMMA - 1)
    return U


def time_step(case, U):
    if case['eqn'] == 'glm_maxwell':
        return case['cfl'] * min(dx_of(case))
    if case['eqn'] == 'euler':
        v, P = prims(U)
        c = (GAMMA * P / U[0]).sqrt()
    else:
        v, c = U[1:4] / U[0], U[0].sqrt()
    return case['cfl'] * torch.stack([dx / (v[a].abs() + c).max() for a, dx in enumerate(dx_of(case))]).min()


def statistics(case, U, fixed):
    G = U
    for a in range(dim_of(case)):
        G = padded(case, G, a, fixed)
    out = []
    for get in (lambda V: V[0], lambda V: prims(V)[1]):
        g, i = get(G), get(U)
        m = i.mean()
        out.append(torch.stack([g.min(), g.max(), m, ((i - m) ** 2).mean().sqrt()]))
    return torch.stack(out)


def solved(case, seed, frames=False):
    """the ghosted final state (z, y, x, S) and the time of a plain case"""
    q = {'euler': 5, 'glm_maxwell': 8, 'shallow_water': 4}[case['eqn']]
    full = initial(case, seed)
    if case['real'] == 'float':
        full = full.to(torch.float32).to(torch.float64)
    fixed = None
    if case['boundary'] == 'fixed':
        fixed = {k: torch.tensor(v, dtype=torch.float64, device=DEV) for k, v in fixed_values(case, full).items()}
    U, stat = constrained(case, full[:q]), full[q:]
    t, seen = 0., []

    def stage(V):
        return derivative(case, V, stat, dt, fixed)

    for _ in range(case['steps']):
        dt = time_step(case, U)
        V = constrained(case, U + dt * stage(U))
        if case['integrator'] == RK2:
            V = constrained(case, .5 * (U + V + dt * stage(V)))
        elif case['integrator'] == RK3:
            V = constrained(case, .75 * U + .25 * (V + dt * stage(V)))
            V = constrained(case, U / 3 + 2 / 3 * (V + dt * stage(V)))
        U, t = V, t + dt
        if frames:
            seen.append((statistics(case, U, fixed), t))
    G = torch.cat([U, stat])
    for a in range(dim_of(case)):
        G = padded(case, G, a, fixed)
    return G.permute(1, 2, 3, 0).contiguous(), float(t), seen


def exact(case, seed):
    if case['kind'] in ('batch', 'serve'):
        out, t, done = [], [], 0
        for i, m in enumerate(members(case)):
            if done < EXACT_GRIDS and m['nx'] * m['ny'] <= EXACT_CELLS:
                U, ti, _ = solved(m, seed * 1009 + i)
                out.append(U)
                done += 1
            else:
                out.append(None)
        return out if case['kind'] == 'batch' else {'U': out, 't': None, 'status': None}
    if case['steps'] * case['nx'] * case['ny'] * case['nz'] * dim_of(case) > 6e9:
        return None
    U, t, seen = solved(case, seed, frames=case['kind'] == 'live')
    if case['kind'] == 'live':
        return {'U': U, 'stats': torch.stack([x for x, _ in seen]), 't': torch.stack([t for _, t in seen])}
    return {'U': U, 't': t}
