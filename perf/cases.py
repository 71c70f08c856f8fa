'''Performance cases of the grid-density path.

Each case is one call that a user's program makes through a public entry
point, on a seeded synthetic molecule of the kind the benchmark and the tests
use: atoms uniform in a cube and at least 1 Angstrom apart, a fixed shell
pattern per atom, three primitives per shell with exponents log-uniform in a
range, unit-normalised contractions, MO coefficients with orthonormal rows,
every MO doubly occupied, grids padded by 5 bohr.

Kinds of case (key ``kind``):
  density   rho and derivatives on a regular grid, inputs kept on the device
            and evaluated again and again (``FusedPlan``)
  points    the same on an atom-centred quadrature grid given as a list of
            points (``FusedPlan`` on a vector grid)
  many      density of a large system with more than 64 MOs (``FusedPlan`` at
            the reduced precisions, ``core.eval_rho`` in FP64)
  gradient  a training step's forward and backward through ``DensityModel``
  batch     many molecules in one graph launch (``BatchPlan``)
  mo, ao    MO or AO values on a grid (``okmi_mo_eval``, ``okmi_ao_eval``)
  api       the whole ``core.rho_compute`` call, host arrays in and out
'''
import ctypes
import math

import numpy
import torch

from orbkit_amd import _native, core, grid
from orbkit_amd.autograd import DensityModel
from orbkit_amd.basis import device_basis
from orbkit_amd.batch import BatchPlan
from orbkit_amd.core import DeviceGrid
from orbkit_amd.fused import FusedPlan
from orbkit_amd.orbitals import AOClass, MOClass
from orbkit_amd.qcinfo import QCinfo

BOHR = 1.0 / 0.52917721092      # bohr per Angstrom
PAD = 5.0                       # bohr between the atoms and a regular grid's faces
CODES = {'': [], 'xyz': [1, 2, 3], 'lap': [4, 5, 6]}   # derivative codes of each ``drv``
ORGANIC = 'sspd'                # shell patterns per atom (comma: taken in turn over the atoms)
MEDIUM = 'ssppdf'
LARGE = 'ssppd,ssppd,ssppd,ssppdf'


# --------------------------------------------------------------------------
# cases
def listed():
  mol = lambda natoms, box, shells, nmo: dict(natoms=natoms, box=box, shells=shells, spherical=True, nmo=nmo,
                                              lo=0.05, hi=1e5)
  box = lambda nx, ny, nz: dict(nx=nx, ny=ny, nz=nz)
  small = dict(mol(3, 4.0, 'spd,spd,ssp', 5), spherical=False, lo=0.1, hi=5000.0)
  medium = mol(20, 12.0, MEDIUM, 40)
  large = mol(200, 30.0, LARGE, 400)
  return [
      # a triatomic on a coarse grid, evaluated inside a loop over new MO
      # coefficients: the launch and its latency
      dict(small, name='small_f64', kind='density', precision='f64', drv='xyz', **box(24, 24, 24)),
      # an orbkit script's call for a small molecule: qc object in, numpy arrays out
      dict(small, name='api_small', kind='api', drv='xyz', **box(50, 50, 50)),
      # the benchmark's headline workload
      dict(medium, name='medium_f64', kind='density', precision='f64', drv='xyz', **box(100, 100, 100)),
      # density and Laplacian terms on a quadrature grid (numerical
      # integration, analysis at chosen points)
      dict(mol(12, 10.0, MEDIUM, 27), name='points_lap_f64', kind='points', precision='f64', drv='lap', nrad=61,
           nang=194),
      # the fast path on a grid whose sides are no multiple of a brick
      dict(medium, name='medium_bf16x6', kind='density', precision='bf16x6', drv='xyz', **box(99, 102, 97)),
      # one step of fitting coefficients, exponents and positions to a target density
      dict(medium, name='gradient_f64', kind='gradient', precision='f64', **box(80, 80, 80)),
      # the same in FP32, ragged grid
      dict(mol(25, 13.0, MEDIUM, 33), name='gradient_f32', kind='gradient', precision='f32', **box(67, 75, 70)),
      # a screening set of organic molecules of uneven size
      dict(name='batch_bf16x6', kind='batch', precision='bf16x6', nmol=24, atoms_lo=5, atoms_hi=60, nmo_lo=8,
           nmo_hi=30, side_lo=32, side_hi=80, shells=ORGANIC, spherical=True, lo=0.05, hi=1e5),
      # a large system, fast path and FP64
      dict(large, name='large_bf16x6', kind='many', precision='bf16x6', drv='xyz', **box(128, 128, 128)),
      dict(large, name='large_f64', kind='many', precision='f64', drv='xyz', **box(96, 101, 104)),
      # every MO on a grid (orbital plots and cube files)
      dict(medium, name='mo_f64', kind='mo', drv='', **box(90, 85, 93)),
      # AO values and first derivatives (a caller's own contraction)
      dict(medium, name='ao_f64', kind='ao', drv='xyz', **box(64, 61, 67)),
  ]


def draw(rng):
  '''One more case of the ranges the listed ones stand for.'''
  logint = lambda a, b: int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

  def box(n):   # ragged sides with about n points in all
    s = n ** (1 / 3)
    sides = [max(4, int(round(s * math.exp(rng.uniform(-0.3, 0.3))))) for _ in range(3)]
    while sides[0] * sides[1] * sides[2] > 1.15 * n:
      sides[sides.index(max(sides))] -= 1
    return dict(zip(('nx', 'ny', 'nz'), sides))

  def molecule(natoms, nmo, shells):
    # box sides about the benchmark's densities of atoms (20 in 12 A, 200 in 30 A)
    c = dict(natoms=natoms, box=round(4.6 * natoms ** (1 / 3) * rng.uniform(0.8, 1.15), 2), shells=shells,
             spherical=True, nmo=nmo, lo=0.05, hi=1e5)
    if 'f' not in shells and rng.random() < 0.3:
      c.update(spherical=False, lo=0.1, hi=5000.0)
    return c

  kind = rng.choice(['density', 'density', 'density', 'points', 'many', 'gradient', 'batch', 'mo', 'ao', 'api'])
  shells = rng.choice([ORGANIC, MEDIUM, 'spd,spd,ssp', 'ssppd'])
  if kind == 'density':
    return dict(molecule(logint(3, 40), logint(2, 64), shells), kind=kind,
                precision=rng.choice(['f64', 'f64', 'bf16x6', 'f32']), drv=rng.choice(['', 'xyz', 'xyz', 'lap']),
                **box(logint(4000, 1000000)))
  if kind == 'points':
    return dict(molecule(logint(2, 20), logint(2, 64), shells), kind=kind, precision='f64',
                drv=rng.choice(['', 'xyz', 'lap']), nrad=rng.randint(20, 75), nang=rng.choice([50, 110, 194, 302]))
  if kind == 'many':
    prec = rng.choice(['f64', 'bf16x6'])
    return dict(molecule(logint(30, 200), logint(65, 400), LARGE), kind=kind, precision=prec,
                drv=rng.choice(['', 'xyz']), **box(logint(20000, 400000)))
  if kind == 'gradient':
    return dict(molecule(logint(4, 25), logint(4, 48), shells), kind=kind, precision=rng.choice(['f64', 'f32']),
                **box(logint(8000, 512000)))
  if kind == 'batch':
    lo = rng.randint(16, 40)
    return dict(kind=kind, precision=rng.choice(['bf16x6', 'f32']), nmol=rng.randint(4, 24), atoms_lo=5,
                atoms_hi=rng.randint(10, 60), nmo_lo=8, nmo_hi=30, side_lo=lo, side_hi=lo + rng.randint(10, 40), shells=ORGANIC, spherical=True,
                lo=0.05, hi=1e5)
  if kind == 'mo':
    return dict(molecule(logint(3, 40), logint(2, 80), shells), kind=kind, drv=rng.choice(['', '', 'xyz']),
                **box(logint(8000, 500000)))
  if kind == 'ao':
    return dict(molecule(logint(3, 25), 8, shells), kind=kind, drv=rng.choice(['', 'xyz', 'lap']),
                **box(logint(8000, 250000)))
  return dict(molecule(logint(3, 20), logint(2, 40), shells), kind=kind, drv=rng.choice(['', 'xyz', 'lap']),
              **box(logint(8000, 150000)))


# --------------------------------------------------------------------------
# inputs from the seed
def _molecule(c, rng):
  '''(positions (natoms, 3), [(atom, l, (3, 2) exponents and coefficients)], C).'''
  pts = []
  while len(pts) < c['natoms']:
    p = rng.uniform(0, c['box'], 3)
    if all(numpy.linalg.norm(p - q) >= 1.0 for q in pts):
      pts.append(p)
  geo = numpy.array(pts) * BOHR
  patterns = c['shells'].split(',')
  shells = []
  for a in range(c['natoms']):
    for t in patterns[a % len(patterns)]:
      l = 'spdf'.index(t)
      al = numpy.sort(numpy.exp(rng.uniform(math.log(c['lo']), math.log(c['hi']), 3)))[::-1]
      co = rng.uniform(0, 1, 3)
      # self-overlap of the contraction of normalised primitives
      s = (2 * numpy.sqrt(al[:, None] * al) / (al[:, None] + al)) ** (l + 1.5)
      shells.append((a, l, numpy.stack([al, co / math.sqrt(co @ s @ co)], axis=1)))
  nao = sum(2 * l + 1 if c['spherical'] else (l + 1) * (l + 2) // 2 for _, l, _ in shells)
  # (the rows of a wide Gaussian matrix, orthonormalised)
  q, _ = numpy.linalg.qr(rng.standard_normal((nao, min(c['nmo'], nao))))
  return geo, shells, numpy.ascontiguousarray(q.T)


def _qc(c, geo, shells, C):
  ao = AOClass()
  for a, l, co in shells:
    ao.append({'atom': a, 'type': 'spdf'[l], 'pnum': len(co), 'coeffs': co})
  if c['spherical']:
    ao.set_lm_dict(p=[1, 0])
  ao.update()
  qc = QCinfo()
  qc.geo_spec = geo
  qc.geo_info = numpy.array([['X', str(i + 1), '0'] for i in range(len(geo))])
  qc.ao_spec = ao
  qc.mo_spec = MOClass([{'coeffs': C[i], 'occ_num': 2.0, 'energy': -1.0 + 0.01 * i, 'sym': '%d.1' % (i + 1)}
                        for i in range(len(C))])
  return qc


def _axes(geo, sides):
  lo, hi = geo.min(axis=0) - PAD, geo.max(axis=0) + PAD
  return [numpy.linspace(lo[i], hi[i], sides[i]) for i in range(3)]


def _quadrature(c, geo):
  '''Radial shells (Becke's map of a midpoint rule) of spread directions on every atom.'''
  k = numpy.arange(c['nang']) + 0.5
  z = 1 - 2 * k / c['nang']
  phi = k * (math.pi * (3 - math.sqrt(5)))
  unit = numpy.stack([numpy.sqrt(1 - z * z) * numpy.cos(phi), numpy.sqrt(1 - z * z) * numpy.sin(phi), z], axis=1)
  t = numpy.cos(math.pi * (numpy.arange(c['nrad']) + 0.5) / c['nrad'])
  r = numpy.minimum((1 + t) / (1 - t), 30.0)
  p = geo[:, None, None, :] + r[None, :, None, None] * unit[None, None, :, :]
  return [numpy.ascontiguousarray(v) for v in p.reshape(-1, 3).T]


def _inputs(c, seed):
  '''(geo, shells, C, axes or point lists) of a one-molecule case.'''
  rng = numpy.random.default_rng(seed)
  geo, shells, C = _molecule(c, rng)
  if c['kind'] == 'points':
    return geo, shells, C, _quadrature(c, geo)
  return geo, shells, C, _axes(geo, [c[k] for k in ('nx', 'ny', 'nz')])


def _batch_inputs(c, seed):
  rng = numpy.random.default_rng(seed)
  # the batch's make-up (atoms, MOs, grid sides) belongs to the case, the molecules to the seed
  shape = numpy.random.default_rng(c['nmol'] * 1000 + c['atoms_hi'])
  out = []
  for _ in range(c['nmol']):
    natoms = int(shape.integers(c['atoms_lo'], c['atoms_hi'] + 1))
    m = dict(c, natoms=natoms, box=4.0 + 0.25 * natoms, nmo=int(shape.integers(c['nmo_lo'], c['nmo_hi'] + 1)))
    side = int(shape.integers(c['side_lo'], c['side_hi'] + 1))
    geo, shells, C = _molecule(m, rng)
    out.append((m, geo, shells, C, _axes(geo, [side] * 3)))
  return out


def _target(axes, geo, dtype):
  '''A target density to fit: a sum of spherical atoms.'''
  pts = _points(axes, True)
  rho = torch.zeros(len(pts), dtype=torch.float64, device=pts.device)
  for g in torch.as_tensor(geo, device=pts.device):
    rho += 1.5 * torch.exp(-1.2 * (pts - g).square().sum(dim=1))
  return rho.to(dtype)


def _device():
  return torch.device('cuda', torch.cuda.current_device())


def _points(axes, regular):
  t = [torch.as_tensor(a, dtype=torch.float64, device=_device()) for a in axes]
  if regular:
    t = torch.meshgrid(*t, indexing='ij')
  return torch.stack([v.reshape(-1) for v in t], dim=1)


def _volume(axes):
  return float(numpy.prod([a[1] - a[0] for a in axes]))


# --------------------------------------------------------------------------
def prepare(case, seed):
  c = case
  if c['kind'] == 'batch':
    mols = _batch_inputs(c, seed)
    plan = BatchPlan([(_qc(m, g, s, C), ax) for m, g, s, C, ax in mols], precision=c['precision'])
    return dict(c=c, plan=plan, stream=torch.cuda.Stream())
  geo, shells, C, axes = _inputs(c, seed)
  qc = _qc(c, geo, shells, C)
  st = dict(c=c, qc=qc, axes=axes)
  if c['kind'] == 'api':
    return st
  if c['kind'] == 'gradient':
    st['model'] = DensityModel(qc, axes, precision=c['precision'])
    st['par'] = st['model'].parameters()
    st['target'] = _target(axes, geo, st['model'].dtype)
    st['d3r'] = _volume(axes)
    return st
  st['basis'] = device_basis(numpy.asarray(qc.geo_spec), qc.ao_spec)
  st['grid'] = DeviceGrid(*axes, regular=c['kind'] != 'points')
  st['codes'] = CODES[c['drv']]
  if c['kind'] in ('mo', 'ao'):
    n, nd = st['grid'].npts, 1 + len(st['codes'])
    st['drv'] = numpy.array([0] + st['codes'], dtype=numpy.intc)
    st['C'] = torch.as_tensor(C, device=_device())
    rows = len(C) if c['kind'] == 'mo' else st['basis'].nao
    st['out'] = torch.empty((nd, rows, n), dtype=torch.float64, device=_device())
    if c['kind'] == 'mo':
      chunk = max(64, min(n, core.WORKSPACE_BYTES // (nd * st['basis'].nao * 8)))
      nbytes = _native.lib().okmi_workspace_bytes(st['basis'].handle, nd, chunk)
      st['ws'] = torch.empty(nbytes // 8 + 1, dtype=torch.float64, device=_device())
    return st
  st['coeffs'], st['occ'] = C, qc.mo_spec.get_occ()
  if not (c['kind'] == 'many' and c['precision'] == 'f64'):
    st['plan'] = FusedPlan(st['basis'], st['grid'], C, st['occ'], st['codes'], precision=c['precision'])
  return st


def run(state):
  s, kind = state, state['c']['kind']
  if kind == 'batch':
    s['plan'].launch(use_graph=True, stream=s['stream'].cuda_stream)
    return [s['plan'].rho, s['plan'].dgrad]
  if kind == 'api':
    grid.set_grid(*s['axes'], is_vector=False)
    drv = s['c']['drv']
    if drv == 'lap':
      return core.rho_compute(s['qc'], laplacian=True)
    return core.rho_compute(s['qc'], drv=list(drv) if drv else None)
  if kind == 'gradient':
    C, alpha, geo = s['par']
    rho = s['model'](C, alpha, geo)
    loss = ((rho - s['target']) ** 2).sum() * s['d3r']
    return [rho.detach()] + list(torch.autograd.grad(loss, (C, alpha, geo)))
  if kind in ('mo', 'ao'):
    L, out, drv = _native.lib(), s['out'], s['drv']
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    where = (s['basis'].handle, ctypes.byref(s['grid'].desc), 0, s['grid'].npts, drv.ctypes.data_as(_native.P_int),
             len(drv))
    dst = (ctypes.c_void_p(out.data_ptr()), out.shape[2])
    if kind == 'ao':
      _native.check(L.okmi_ao_eval(*where, _native.OKMI_F64, *dst, stream), 'okmi_ao_eval')
    else:
      _native.check(L.okmi_mo_eval(*where, ctypes.c_void_p(s['C'].data_ptr()), s['C'].shape[0], *dst,
                                   ctypes.c_void_p(s['ws'].data_ptr()), s['ws'].numel() * 8, stream), 'okmi_mo_eval')
    return out
  if 'plan' in s:
    s['plan'].launch()
    return [s['plan'].rho, s['plan'].delta] if s['codes'] else s['plan'].rho
  rho, delta, _ = core.eval_rho(s['basis'], s['grid'], s['coeffs'], s['occ'], s['codes'], device=True)
  return [rho, delta] if s['codes'] else rho


# --------------------------------------------------------------------------
def _row_terms(l, spherical):
  '''AO rows of a shell as polynomials {(lx, ly, lz): factor}, to be
  multiplied by sum_p c_p N_p exp(-alpha_p r^2) with N_p = (2/pi)^(3/4) 2^l
  alpha_p^((2l+3)/4): normalised Cartesian components, or real solid harmonics
  in the order m = 0, 1, -1, 2, -2, ... (p: x, y, z).'''
  if l == 0:
    return [{(0, 0, 0): 1.0}]
  if l == 1:
    return [{(1, 0, 0): 1.0}, {(0, 1, 0): 1.0}, {(0, 0, 1): 1.0}]
  if l == 2 and not spherical:
    q = 1 / math.sqrt(3)
    return [{(2, 0, 0): q}, {(0, 2, 0): q}, {(0, 0, 2): q}, {(1, 1, 0): 1.0}, {(1, 0, 1): 1.0}, {(0, 1, 1): 1.0}]
  if l == 2:
    q = 1 / math.sqrt(12)
    return [{(0, 0, 2): 2 * q, (2, 0, 0): -q, (0, 2, 0): -q}, {(1, 0, 1): 1.0}, {(0, 1, 1): 1.0},
            {(2, 0, 0): 0.5, (0, 2, 0): -0.5}, {(1, 1, 0): 1.0}]
  q0, q1, q3 = 1 / math.sqrt(60), 1 / math.sqrt(40), 1 / math.sqrt(24)
  return [{(0, 0, 3): 2 * q0, (2, 0, 1): -3 * q0, (0, 2, 1): -3 * q0},
          {(1, 0, 2): 4 * q1, (3, 0, 0): -q1, (1, 2, 0): -q1},
          {(0, 1, 2): 4 * q1, (2, 1, 0): -q1, (0, 3, 0): -q1},
          {(2, 0, 1): 0.5, (0, 2, 1): -0.5}, {(1, 1, 1): 1.0},
          {(3, 0, 0): q3, (1, 2, 0): -3 * q3}, {(2, 1, 0): 3 * q3, (0, 3, 0): -q3}]


def _polynomial(terms, X, drv=()):
  '''Value of the polynomial (differentiated along each axis of ``drv``) at X (3, n).'''
  v = 0.0
  for e, f in terms.items():
    e = list(e)
    for a in drv:
      f *= e[a]
      e[a] -= 1
    if f:
      v = v + f * X[0] ** e[0] * X[1] ** e[1] * X[2] ** e[2]
  return v


def _ao(c, shells, alpha, geo, pts, codes):
  '''AO values of each derivative code: a list of (nao, n) tensors in 64 bits.'''
  out = [[] for _ in codes]
  k = 0
  for a, l, co in shells:
    al = alpha[k:k + len(co)]
    k += len(co)
    X = (pts - geo[a]).T
    r2 = X.square().sum(dim=0)
    d = torch.as_tensor(co[:, 1].copy(), device=pts.device) * ((2 / math.pi) ** 0.75 * 2 ** l) * al ** ((2 * l + 3) / 4)
    e = d[:, None] * torch.exp(-al[:, None] * r2)
    S0, S1, S2 = e.sum(dim=0), (-2 * al[:, None] * e).sum(dim=0), (4 * al[:, None] ** 2 * e).sum(dim=0)
    for terms in _row_terms(l, c['spherical']):
      p = _polynomial(terms, X)
      for rows, code in zip(out, codes):
        i = (code - 1) % 3
        if code == 0:
          rows.append(p * S0)
        elif code <= 3:
          rows.append(_polynomial(terms, X, (i,)) * S0 + X[i] * p * S1)
        else:
          rows.append(_polynomial(terms, X, (i, i)) * S0 + 2 * X[i] * _polynomial(terms, X, (i,)) * S1 + p * S1 +
                      X[i] ** 2 * p * S2)
  return [torch.stack([r + torch.zeros_like(S0) for r in rows]) for rows in out]


def _tensors(shells, geo, C):
  t = lambda v: torch.as_tensor(numpy.ascontiguousarray(v), device=_device())
  return t(numpy.concatenate([co[:, 0] for _, _, co in shells])), t(geo), t(C)


def _chunk(nao, nsets):
  return max(1024, int(2e9 / (8 * nao * nsets)))


def _density(c, geo, shells, C, pts, codes):
  '''rho (n,) and the derivative rows (len(codes), n) in 64 bits.'''
  alpha, g, Ct = _tensors(shells, geo, C)
  sets = sorted({0} | set(codes) | ({1, 2, 3} if any(k > 3 for k in codes) else set()))
  rho = torch.empty(len(pts), dtype=torch.float64, device=pts.device)
  delta = torch.empty((len(codes), len(pts)), dtype=torch.float64, device=pts.device)
  step = _chunk(Ct.shape[1], len(sets))
  for p in range(0, len(pts), step):
    phi = dict(zip(sets, (Ct @ A for A in _ao(c, shells, alpha, g, pts[p:p + step], sets))))
    rho[p:p + step] = 2 * phi[0].square().sum(dim=0)
    for row, k in zip(delta, codes):
      v = phi[0] * phi[k]
      if k > 3:
        v = v + phi[k - 3].square()
      row[p:p + step] = 4 * v.sum(dim=0)
  return rho, delta


def exact(case, seed):
  c = case
  if c['kind'] == 'batch':
    got = [_density(m, g, s, C, _points(ax, True), [1, 2, 3]) for m, g, s, C, ax in _batch_inputs(c, seed)]
    return [[r for r, _ in got], [d for _, d in got]]
  geo, shells, C, axes = _inputs(c, seed)
  pts = _points(axes, c['kind'] != 'points')
  if c['kind'] == 'gradient':
    alpha, g, Ct = _tensors(shells, geo, C)
    dtype = torch.float64 if c['precision'] == 'f64' else torch.float32
    par = [v.to(dtype).double().requires_grad_() for v in (Ct, alpha, g)]
    target, d3r = _target(axes, geo, dtype).double(), _volume(axes)
    step = _chunk(par[0].shape[1], 24)
    rho, grads = [], None
    for p in range(0, len(pts), step):
      r = 2 * (par[0] @ _ao(c, shells, par[1], par[2], pts[p:p + step], [0])[0]).square().sum(dim=0)
      new = torch.autograd.grad(((r - target[p:p + step]) ** 2).sum() * d3r, par)
      grads = new if grads is None else [a + b for a, b in zip(grads, new)]
      rho.append(r.detach())
    return [torch.cat(rho)] + list(grads)
  codes = CODES[c['drv']]
  if c['kind'] in ('mo', 'ao'):
    alpha, g, Ct = _tensors(shells, geo, C)
    parts = []
    for q in pts.split(_chunk(Ct.shape[1], 2 * (1 + len(codes)))):
      parts.append(torch.stack([Ct @ A if c['kind'] == 'mo' else A for A in _ao(c, shells, alpha, g, q, [0] + codes)]))
    return torch.cat(parts, dim=2)
  rho, delta = _density(c, geo, shells, C, pts, codes)
  if c['kind'] == 'api':
    n = tuple(len(a) for a in axes)
    out = (rho.reshape(n), delta.reshape((len(codes),) + n))
    return out[0] if not codes else out if c['drv'] != 'lap' else out + (out[1].sum(dim=0),)
  return [rho, delta] if codes else rho


# --------------------------------------------------------------------------
def _live(shells, spherical, geo, axes, regular):
  '''Share of (AO row, point) and of (primitive, point) pairs with
  exp(-alpha r^2) above 1e-24, from 2,000 of the points: the rest adds
  nothing to a density in 64 bits.'''
  rng = numpy.random.default_rng(0)
  n = 2000
  if regular:
    p = numpy.stack([rng.choice(a, n) for a in axes], axis=1)
  else:
    p = numpy.stack(axes, axis=1)[rng.integers(0, len(axes[0]), n)]
  r2 = ((p[:, None, :] - geo) ** 2).sum(axis=2)
  rows = prims = 0.0
  for a, l, co in shells:
    rows += (2 * l + 1 if spherical else (l + 1) * (l + 2) // 2) * float((co[:, 0].min() * r2[:, a] < 55.0).mean())
    prims += float((co[:, 0] * r2[:, a, None] < 55.0).mean(axis=0).sum())
  return rows, prims


def work(case):
  '''Bytes: inputs read once, outputs written once.  Flops per point: 2 NMO per
  AO row in reach and AO set for the contraction (three such products for a
  gradient), 20 per primitive in reach (an exponential and its sums).'''
  c = case
  if c['kind'] == 'batch':
    bytes_ = flops = 0.0
    for m, geo, shells, C, axes in _batch_inputs(c, 0):
      n = len(axes[0]) ** 3
      rows, prims = _live(shells, True, geo, axes, True)
      bytes_ += 8.0 * (4 * n + C.size)
      flops += n * (2.0 * len(C) * rows * 4 + 20 * prims)
    return {'bytes': bytes_, 'flops': flops}
  geo, shells, C, axes = _inputs(c, 0)
  regular = c['kind'] != 'points'
  n = float(len(axes[0]) if not regular else len(axes[0]) * len(axes[1]) * len(axes[2]))
  rows, prims = _live(shells, c['spherical'], geo, axes, regular)
  if c['kind'] == 'gradient':
    size = 8 if c['precision'] == 'f64' else 4
    return {'bytes': size * (3.0 * n + 2 * C.size), 'flops': n * (4 * 2.0 * len(C) * rows + 40 * prims)}
  sets = {'': 1, 'xyz': 4, 'lap': 4 if c['kind'] in ('ao', 'mo') else 7}[c['drv']]
  nout = {'': 1, 'xyz': 4, 'lap': 4}[c['drv']]
  inputs = 8.0 * (C.size + sum(len(a) for a in axes))
  if c['kind'] == 'ao':
    return {'bytes': inputs + 8.0 * n * sets * C.shape[1], 'flops': n * (20.0 * prims + 2 * sets * rows)}
  if c['kind'] == 'mo':
    return {'bytes': inputs + 8.0 * n * sets * len(C), 'flops': n * (20.0 * prims + 2.0 * len(C) * rows * sets)}
  return {'bytes': inputs + 8.0 * n * nout, 'flops': n * (20.0 * prims + 2.0 * len(C) * rows * sets)}
