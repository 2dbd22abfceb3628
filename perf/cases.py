"""What a program has this framework do, as cases that can be timed and compared: one frequency point's parts and
whole points, from a strip of a few hundred unknowns to a 20 000-unknown factor, in both precisions.

Kinds of case (the public entry point each calls):
  factor  gpu.HipBackend.factor_device + solve_device: the dense complex LU of an equilibrated Z and the port solves
  solve   gpu.HipBackend.solve_device with a factor already there: the preconditioner of every refinement iteration
          (trans 1: Z X = R; trans 0: its transpose)
  refine  linalg.gmres_batched: the FP64 refinement of a point on the complex64 factor of a nearby frequency, products
          with the FP64 Z (device.zgemm_nk), to the solver's tolerance of 1e-6
  fill    Simulation.fast.fill: a frequency's whole Z of a board (Green's tables, far field, near field, vias), stored
          as complex128, or as complex64 (the lean path)
  matvec  Simulation.fast.matvec_exact: the FP64 operator without Z (the lean path's refinement product)
  point   Simulation.sparams: a whole frequency point, S out
  batch   batch.SweepBatch: many points of boards of uneven size in mixed precision, S of each out

Sizes are those of the package's boards and of bench.py's configurations (a strip of about 900 unknowns, the 4-layer
board of 7799, the coupled lines of about 3500, boards up to 20 000) and others between them. Matrices of the first
three kinds are made here, in the form the fill gives them: unit diagonal, coupling that falls off with distance along
traces and turns with the wavenumber, and some rows exchanged so that pivots leave the diagonal. Boards are the
package's own with permittivities and frequencies drawn from the seed.

A complex64 factor's solutions are complex64 numbers in a complex128 tensor, and a refinement to 1e-6 or a mixed
point's S is good to about six digits: these come out as complex64, the type that holds what was computed; everything
computed in FP64 throughout comes out as complex128.
"""
import math

import numpy as np
import torch

from mom25d_amd import boards, device as dv
from mom25d_amd.batch import SweepBatch
from mom25d_amd.gpu import HipBackend
from mom25d_amd.linalg import gmres_batched
from mom25d_amd.multilayer import Layer, LayerStack
from mom25d_amd.sim import Simulation

MM = 1e-3
EXACT_N = 9000                     # the largest system that is solved again in plain FP64 for comparison


# ---- the cases ----------------------------------------------------------------------------------------------
def listed():
    return [
        # the smallest factor a backend call meets in earnest: a strip's few hundred unknowns, two ports
        dict(name='factor_c64_905', kind='factor', n=905, k=2, dtype='c64'),
        # the complex64 factor of the 4-layer benchmark board, four ports
        dict(name='factor_c64_7799', kind='factor', n=7799, k=4, dtype='c64'),
        # the largest board of the serving configuration
        dict(name='factor_c64_20000', kind='factor', n=20000, k=4, dtype='c64'),
        # the plain FP64 path's factor of the same board, and where a complex64 one does not converge
        dict(name='factor_c128_7799', kind='factor', n=7799, k=4, dtype='c128'),
        # one application of a kept factor in a refinement
        dict(name='solve_c64_7799', kind='solve', n=7799, k=4, dtype='c64', trans=1),
        # an FP64 factor against many right-hand sides, an odd size, the transposed system
        dict(name='solve_c128_3001', kind='solve', n=3001, k=7, dtype='c128', trans=0),
        # a sweep's ordinary point: GMRES on the factor of the last frequency
        dict(name='refine_7799', kind='refine', n=7799, k=4),
        # the fill of the benchmark board
        dict(name='fill_board', kind='fill', board='seeded', dmax=0.25, ncross=3, dtype='c128'),
        # the lean path's fill and product on the coupled-line board
        dict(name='fill_lean_lines', kind='fill', board='lines', dmax=0.25, ncross=4, dtype='c64'),
        dict(name='matvec_lines', kind='matvec', board='lines', dmax=0.25, ncross=4, k=4),
        # a whole FP64 point of the strip (one of the 101 linear points of its sweep)
        dict(name='point_strip', kind='point', board='strip', dmax=0.3, ncross=4, precision='double'),
        # a batch of points: coupled lines meshed at three densities, eight frequencies each, mixed precision
        dict(name='batch_lines', kind='batch', board='lines', dmax=0.3, ncross=3, boards=3, points=8),
    ]


def draw(rng):
    """One more case of the same kinds and ranges."""
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    kind = rng.choice(['factor', 'factor', 'solve', 'solve', 'refine', 'fill', 'fill', 'matvec', 'point', 'batch'])
    board = rng.choice(['strip', 'lines', 'seeded'])
    mesh = dict(board=board, dmax=round(rng.uniform(0.25, 0.6), 3), ncross=rng.choice([2, 3, 4]))
    if board == 'seeded':
        mesh['ncross'] = min(3, mesh['ncross'])        # no board above the benchmark's size
    if kind == 'factor':
        dtype = rng.choice(['c64', 'c128'])
        return dict(kind=kind, n=size(300, 18000 if dtype == 'c64' else 8500), k=rng.randint(1, 8), dtype=dtype)
    if kind == 'solve':
        return dict(kind=kind, n=size(300, 12000), k=rng.randint(1, 8), dtype=rng.choice(['c64', 'c128']),
                    trans=rng.choice([0, 1]))
    if kind == 'refine':
        return dict(kind=kind, n=size(300, 8500), k=rng.randint(1, 8))
    if kind == 'fill':
        return dict(kind=kind, dtype=rng.choice(['c64', 'c128']), **mesh)
    if kind == 'matvec':
        return dict(kind=kind, k=rng.randint(1, 8), **mesh)
    if kind == 'point':
        mesh['board'] = rng.choice(['strip', 'lines'])
        return dict(kind=kind, precision='double', **mesh)
    mesh['board'] = rng.choice(['strip', 'lines'])
    return dict(kind='batch', boards=rng.randint(1, 3), points=rng.randint(2, 8), **mesh)


# ---- matrices in the form of an equilibrated Z ------------------------------------------------------------------
def _generator(seed, extra=0):
    return torch.Generator('cuda').manual_seed(1000003 * int(seed) + extra)


def _system(n, seed, waves=(5.0,)):
    """[Z] (n x n complex128, unit diagonal) at each wavenumber: cells along n / 300 traces, neighbours coupled about
    half as strongly as a cell to itself, the rest falling off as distance^-1.5 and turning with the wavenumber; a
    random part; every eighth pair of rows three apart exchanged."""
    g, dev, f64 = _generator(seed), 'cuda', torch.float64
    ntr = max(1, n // 300)
    i = torch.arange(n, device=dev)
    t = (i * ntr) // n
    first = torch.searchsorted(t, torch.arange(ntr, device=dev))
    step = 1.0 / math.sqrt(n)
    p = (torch.rand(ntr, 2, generator=g, device=dev, dtype=f64) * 2 - 1)[t]
    p[i, t % 2] += (i - first[t]) * step
    out = [torch.empty((n, n), dtype=torch.complex128, device=dev) for _ in waves]
    for a in range(0, n, 2048):
        b = min(n, a + 2048)
        R = torch.sqrt((p[a:b, None, 0] - p[None, :, 0]) ** 2 + (p[a:b, None, 1] - p[None, :, 1]) ** 2)
        mag = 0.5 / (1 + R / step) ** 1.5 * torch.where((t[a:b, None] - t[None, :]) % 2 == 0, 1.0, 0.25)
        noise = torch.randn(b - a, n, generator=g, device=dev, dtype=torch.complex128) * (0.5 / math.sqrt(n))
        for Z, k in zip(out, waves):
            Z[a:b] = torch.polar(mag, -k * R) + noise
    ph = 0.1 * torch.randn(n, generator=g, device=dev, dtype=f64)
    order = torch.arange(n, device=dev)
    move = torch.nonzero(torch.rand(n // 8, generator=g, device=dev) < 0.5).ravel() * 8
    move = move[move + 3 < n]
    order[move], order[move + 3] = move + 3, move
    for j, Z in enumerate(out):
        Z[i, i] = torch.polar(torch.ones_like(ph), ph)
        out[j] = Z[order]
    return out


def _ports(n, k, seed):
    """Port excitations: one entry a column, as a via port's."""
    R = torch.zeros((n, k), dtype=torch.complex128, device='cuda')
    rows = torch.randperm(n, generator=_generator(seed, 1), device='cuda')[:k]
    R[rows, torch.arange(k, device='cuda')] = 1.0
    return R


def _dense(n, k, seed):
    """Right-hand sides as a refinement iteration has them: every entry filled."""
    return torch.randn(n, k, generator=_generator(seed, 2), device='cuda', dtype=torch.complex128)


_DTYPE = {'c64': torch.complex64, 'c128': torch.complex128}


# ---- boards ------------------------------------------------------------------------------------------------------
def _board(case, seed=None, scale=1.0, mesh_only=False, precision='auto'):
    """The case's board (its mesh fixed by the case; every layer's permittivity drawn within 5 % from the seed)."""
    make = {'strip': boards.microstrip, 'lines': boards.coupled_lines, 'seeded': boards.seeded_board}[case['board']]
    st, shapes, ports, vias, kw = make(dmax=case['dmax'] * scale * MM, ncross=case['ncross'])
    if seed is not None:
        rng = np.random.default_rng(seed)
        st = LayerStack([Layer(l.h, l.er * rng.uniform(0.95, 1.05), l.tand) for l in st.layers])
    return Simulation(st, shapes, ports, vias, verbose=False, mesh_only=mesh_only, precision=precision, **kw)


def _freqs(seed, n, lo=1e9, hi=8e9):
    """A sweep's frequencies, log-spaced from a start drawn from the seed."""
    f0 = lo * np.random.default_rng([seed, 7]).uniform(1.0, 1.1)
    return [float(f) for f in np.geomspace(f0, hi, n)]


_SCALES = (1.0, 1.25, 1.6)         # a batch's boards: mesh densities


# ---- one case ----------------------------------------------------------------------------------------------------
def prepare(case, seed):
    kind = case['kind']
    st = dict(case)
    if kind == 'factor':
        st['Z'] = _system(case['n'], seed)[0].to(_DTYPE[case['dtype']])
        st['R'], st['backend'] = _ports(case['n'], case['k'], seed), HipBackend()
    elif kind == 'solve':
        st['R'], st['backend'] = _dense(case['n'], case['k'], seed), HipBackend()
        st['backend'].factor_device(_system(case['n'], seed)[0].to(_DTYPE[case['dtype']]))
    elif kind == 'refine':
        Z0, st['Z'] = _system(case['n'], seed, (5.0, 13.0))
        st['R'], st['backend'] = _ports(case['n'], case['k'], seed), HipBackend()
        st['backend'].factor_device(Z0.to(torch.complex64))
    elif kind in ('fill', 'matvec', 'point'):
        st['sim'] = _board(case, seed, precision=case.get('precision', 'auto'))
        st['freqs'], st['at'] = _freqs(seed, 16), 0
        if kind == 'matvec':
            st['sim'].fast.fill(st['freqs'][0], torch.complex64)
            st['X'] = _dense(st['sim'].Ne + st['sim'].Nv, case['k'], seed)
    else:
        sims = [_board(case, seed, s) for s in _SCALES[:case['boards']]]
        st['points'] = [(s, f) for s in sims for f in _freqs(seed, case['points'])]
    return st


def _next_frequency(st):
    """A sweep goes on: every pass is at the next of its frequencies."""
    f = st['freqs'][st['at'] % len(st['freqs'])]
    st['at'] += 1
    return f


def run(st):
    kind = st['kind']
    if kind == 'factor':
        st['backend'].factor_device(st['Z'].clone())       # in place: Z is kept, as for the refinement's products
        return st['backend'].solve_device(st['R']).to(_DTYPE[st['dtype']])
    if kind == 'solve':
        return st['backend'].solve_device(st['R'], trans=st['trans']).to(_DTYPE[st['dtype']])
    if kind == 'refine':
        Z, backend = st['Z'], st['backend']
        X, _ = gmres_batched(lambda V: dv.zgemm_nk(Z, V), st['R'], M=backend.solve_device, rtol=1e-6, restart=60,
                             maxiter=1)
        return X.to(torch.complex64)
    if kind == 'fill':
        return st['sim'].fast.fill(_next_frequency(st), _DTYPE[st['dtype']])
    if kind == 'matvec':
        return st['sim'].fast.matvec_exact(st['X'])
    if kind == 'point':
        return st['sim'].sparams(_next_frequency(st))
    return [S.astype(np.complex64) for S in SweepBatch(st['points']).run()]


def exact(case, seed):
    """The solutions of the made systems by plain FP64 LU. The boards' cases have none: their values are a whole
    Green's-function and moment code's."""
    kind = case['kind']
    if kind not in ('factor', 'solve', 'refine') or case['n'] > EXACT_N:
        return None
    if kind == 'refine':
        Z = _system(case['n'], seed, (5.0, 13.0))[1]
    else:
        Z = _system(case['n'], seed)[0].to(_DTYPE[case['dtype']]).to(torch.complex128)
    R = (_dense if kind == 'solve' else _ports)(case['n'], case['k'], seed)
    if kind == 'solve' and case['trans'] == 0:
        Z = Z.T.contiguous()
    return torch.linalg.solve(Z, R)


# ---- what a pass cannot do without -------------------------------------------------------------------------------
_SIZES = {}


def _size(case, scale=1.0):
    """(unknowns, triangles) of the case's board."""
    key = (case['board'], case['dmax'] * scale, case['ncross'])
    if key not in _SIZES:
        sim = _board(case, scale=scale, mesh_only=True)
        _SIZES[key] = (sim.Ne + sim.Nv, len(sim.rwg.tris))
    return _SIZES[key]


KERNEL_FLOPS = 40                  # one kernel value at a distance: the distance, two complex interpolations, 1 / r


def _fill_work(n, nt, item):
    """Z written once; a kernel value for each of the nt (nt + 1) / 2 triangle pairs, an entry's four terms of each of
    the n (n + 1) / 2 pairs of unknowns."""
    return item * n * n, KERNEL_FLOPS * nt * nt / 2 + 40.0 * n * n / 2


def work(case):
    kind, k = case['kind'], case.get('k', 0)
    item = 8 if case.get('dtype') == 'c64' else 16
    if kind in ('factor', 'solve', 'refine'):
        n = case['n']
        if kind == 'factor':               # Z read, its factor written; the right-hand sides read, solutions written
            return dict(bytes=2.0 * item * n * n + 32.0 * n * k, flops=8 / 3 * n ** 3 + 8.0 * n * n * k)
        if kind == 'solve':                # the factor read once
            return dict(bytes=item * n * n + 32.0 * n * k, flops=8.0 * n * n * k)
        its = 11                           # iterations these systems take: the FP64 Z and the complex64 factor each
        return dict(bytes=its * (16.0 + 8.0) * n * n, flops=its * 16.0 * n * n * k)
    if kind == 'batch':
        b = f = 0.0
        for s in _SCALES[:case['boards']]:
            n, nt = _size(case, s)
            fb, ff = _fill_work(n, nt, 16)             # FP64 Z, its complex64 factor, two refinement iterations
            b += case['points'] * (fb + 8.0 * n * n + 2 * 24.0 * n * n)
            f += case['points'] * (ff + 8 / 3 * n ** 3)
        return dict(bytes=b, flops=f)
    n, nt = _size(case)
    if kind == 'matvec':                   # a kernel value for every triangle pair, applied to k columns; X in, Y out
        return dict(bytes=32.0 * n * k, flops=nt * nt * (KERNEL_FLOPS / 2 + 24.0 * k))
    b, f = _fill_work(n, nt, item)
    if kind == 'point':                    # Z written, read by the factor and its factor written
        return dict(bytes=3 * b, flops=f + 8 / 3 * n ** 3)
    return dict(bytes=b, flops=f)
