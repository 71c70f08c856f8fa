'''FP64 kernels that list the shells in reach of a tile (densities, MO and AO
values) against the oracle, at the sizes where their splits change: MO counts
around whole groups of 4 and around the groups of 64 of a launch, more shells in
reach than a list holds (256), classes with one to three shells left over, one
to nine primitives, every angular momentum, Cartesian and real spherical rows
(g: general row maps), odd numbers of points.  Bar: that of every FP64 path
(max|gpu - oracle| <= 1e-12 max|oracle|).
'''
import numpy
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-12


def _molecule(natoms, types, spherical, nmo, seed=1):
  from orbkit_amd.orbitals import AOClass, MOClass
  from orbkit_amd.qcinfo import QCinfo
  rng = numpy.random.default_rng(seed)
  qc = QCinfo()
  qc.geo_spec = rng.uniform(-4, 4, (natoms, 3))
  qc.geo_info = numpy.array([['X', str(i + 1), '0'] for i in range(natoms)])
  ao = AOClass()
  for at in range(natoms):
    for l in types:
      pnum = int(rng.choice([1, 3, 4, 5, 9]))
      co = numpy.stack([numpy.sort(numpy.exp(rng.uniform(-2, 5, pnum)))[::-1], rng.uniform(0.2, 1, pnum)], axis=1)
      ao.append({'atom': at, 'type': l, 'pnum': pnum, 'coeffs': co})
  if spherical:
    ao.set_lm_dict(p=[1, 0])
  ao.update()
  nao = sum(2 * 'spdfg'.index(l) + 1 if spherical else ('spdfg'.index(l) + 1) * ('spdfg'.index(l) + 2) // 2
            for l in types) * natoms
  C = rng.standard_normal((nmo, nao)) / nao ** 0.5
  qc.ao_spec = ao
  qc.mo_spec = MOClass([{'coeffs': C[i], 'occ_num': float(rng.uniform(0.5, 2)), 'energy': -1.0 + 0.01 * i,
                         'sym': '%d.1' % (i + 1)} for i in range(nmo)])
  return qc


def _check(qc, points, **kw):
  import torch
  if not torch.cuda.is_available():
    pytest.skip('no HIP device')
  from orbkit_amd import core, grid
  from oracle import core_oracle
  rng = numpy.random.default_rng(2)
  if points is None:   # a regular grid whose sides are no multiples of a brick
    axes = [numpy.linspace(-5, 5, n) for n in (5, 9, 6)]
  else:
    axes = list(rng.uniform(-5, 5, (3, points)))
  grid.set_grid(*axes, is_vector=points is not None)
  got = core.rho_compute(qc, **kw)
  want = core_oracle.rho_compute(qc, *axes, points is not None, **kw)
  for a, b in zip(*[v if isinstance(v, tuple) else (v,) for v in (got, want)]):
    assert a.shape == b.shape
    assert rel_err(a, b) <= TOL


@pytest.mark.parametrize('points', [None, 1, 131])
@pytest.mark.parametrize('drv', [None, ['x', 'y', 'z'], ['xx', 'yy', 'zz'], ['xy', 'z']])
@pytest.mark.parametrize('nmo', [1, 4, 5, 41, 64, 65, 130])
def test_density(nmo, drv, points):
  print('case', nmo, drv, points, flush=True)
  _check(_molecule(7, 'sspdf', True, nmo), points, drv=drv)


@pytest.mark.parametrize('drv', [None, ['x', 'y', 'z'], ['xx', 'yy', 'zz']])
@pytest.mark.parametrize('spherical,types,natoms', [(True, 'spdfg', 3), (False, 'spdfg', 2), (False, 'spd', 1),
                                                    (True, 'ssssp', 60)])
def test_shells(natoms, types, spherical, drv):
  print('case', natoms, types, spherical, drv, flush=True)
  _check(_molecule(natoms, types, spherical, 6), 100, drv=drv)


@pytest.mark.parametrize('kind', ['calc_mo', 'calc_ao'])
@pytest.mark.parametrize('points', [None, 63, 257])
@pytest.mark.parametrize('drv', [None, ['x', 'zz', 'yz'], ['z', 'y']])
@pytest.mark.parametrize('spherical,nmo', [(True, 3), (False, 67)])
def test_values(spherical, nmo, drv, points, kind):
  print('case', spherical, nmo, drv, points, kind, flush=True)
  _check(_molecule(4, 'spdfg', spherical, nmo), points, drv=drv, **{kind: True})
