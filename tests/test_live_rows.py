'''AO sets of a tile's live chunks through the staged FP64 density: shells of every angular momentum, one to nine primitives,
Cartesian and real spherical rows (g: general row maps), regular grids padded to bricks and
vector grids that end inside a tile, against the FP64 kernel that evaluates
the shells in its registers, at the bar of every FP64 path.
'''
import numpy
import pytest

pytestmark = pytest.mark.gpu


def _basis(spherical):
  from orbkit_amd.basis import device_basis
  from orbkit_amd.orbitals import AOClass
  rng = numpy.random.default_rng(5 + spherical)
  geo = rng.uniform(-6, 6, (9, 3))
  ao = AOClass()
  for at in range(len(geo)):
    for l, pnum in zip('spdfg', rng.permutation([1, 3, 4, 5, 9])):
      co = numpy.stack([numpy.sort(numpy.exp(rng.uniform(-2, 6, pnum)))[::-1], rng.uniform(0.2, 1, pnum)], axis=1)
      ao.append({'atom': at, 'type': str(l), 'pnum': int(pnum), 'coeffs': co})
  if spherical:
    ao.set_lm_dict(p=[1, 0])
  ao.update()
  return device_basis(geo, ao)


@pytest.mark.parametrize('points', [None, 65, 700])
@pytest.mark.parametrize('codes', [[], [2, 1, 3], [5, 1]])
@pytest.mark.parametrize('spherical', [False, True])
def test_live_rows(spherical, codes, points):
  import torch
  if not torch.cuda.is_available():
    pytest.skip('no HIP device')
  from orbkit_amd import core
  from orbkit_amd.core import DeviceGrid
  basis = _basis(spherical)
  rng = numpy.random.default_rng(3)
  C = rng.standard_normal((70, basis.nao)) / basis.nao ** 0.5
  occ = rng.uniform(0.5, 2, 70)
  if points is None:
    g = DeviceGrid(numpy.linspace(-9, 9, 10), numpy.linspace(-8, 9, 13), numpy.linspace(-9, 7, 7), regular=True)
  else:
    g = DeviceGrid(*rng.uniform(-9, 9, (3, points)), regular=False)
  print('case', spherical, codes, points, flush=True)
  ref = core.eval_rho(basis, g, C, occ, codes)[:2]
  got = core.eval_rho(basis, g, C, occ, codes, staged=True)
  for a, b in list(zip(got, ref))[:2 if codes else 1]:
    assert numpy.linalg.norm(a - b) <= 1e-12 * numpy.linalg.norm(b)
