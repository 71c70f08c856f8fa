'''The split-bf16 many-MO path for rho and rho with first derivatives against
the FP64 path: MO counts at the edges of its blocks (up to five tiles of 16,
spread evenly, the last one ragged), regular grids padded to bricks, vector
grids that end inside a tile, and workspaces from the whole grid down to the
smallest one accepted.

Bars: norm-wise, those of the path's other precision tests (bf16x6 2.5e-7,
bf16x3 2e-5); passes of different length give the same FP32 sums, whose FP64
reduction is the same too: equal results.
'''
import re

import numpy
import pytest

pytestmark = pytest.mark.gpu

TOL = {'bf16x6': 2.5e-7, 'bf16x3': 2e-5}


@pytest.fixture(scope='module')
def mol():
  import torch
  if not torch.cuda.is_available():
    pytest.skip('no HIP device')
  from orbkit_amd import workloads
  from orbkit_amd.basis import device_basis
  qc, axes, _ = workloads.make('medium', npts_side=16, nmo=177)
  return device_basis(qc.geo_spec, qc.ao_spec), qc.mo_spec.get_coeffs(), axes


def _grid(axes, points):
  from orbkit_amd.core import DeviceGrid
  if points is None:
    return DeviceGrid(axes[0][:13], axes[1][2:9], axes[2][:10], regular=True)
  rng = numpy.random.default_rng(points)
  return DeviceGrid(*[rng.uniform(a[0], a[-1], points) for a in axes], regular=False)


@pytest.mark.parametrize('points', [None, 1, 129, 1777])
@pytest.mark.parametrize('codes', [[], [1, 2, 3]])
@pytest.mark.parametrize('nmo,prec', [(65, 'bf16x6'), (80, 'bf16x6'), (81, 'bf16x3'), (112, 'bf16x6'), (161, 'bf16x6'),
                                      (177, 'bf16x3')])
def test_split_blocks(mol, nmo, prec, codes, points):
  from orbkit_amd import core
  from orbkit_amd.fused import rho_fused
  basis, C, axes = mol
  occ = numpy.linspace(0.5, 2.0, nmo)
  g = _grid(axes, points)
  print('case', nmo, prec, codes, points, flush=True)
  rho, delta = rho_fused(basis, g, C[:nmo], occ, codes, prec)
  ref, dref, _ = core.eval_rho(basis, g, C[:nmo], occ, codes)
  for got, want in [(rho, ref), (delta, dref)][:2 if codes else 1]:
    e = numpy.linalg.norm(got - want) / numpy.linalg.norm(want)
    assert e <= TOL[prec], e


@pytest.mark.parametrize('points', [None, 301])
@pytest.mark.parametrize('codes', [[], [3, 1]])
def test_split_workspaces(mol, codes, points):
  import torch
  from orbkit_amd import _native
  from orbkit_amd.fused import FusedPlan
  basis, C, axes = mol
  plan = FusedPlan(basis, _grid(axes, points), C[:112], numpy.full(112, 2.0), codes, 'bf16x6')
  plan.launch()
  whole = plan.result()
  plan.ws = plan.ws[:64]
  with pytest.raises(Exception, match='too small') as e:
    plan.launch()
  need = int(re.search(r'need at least (\d+)', str(e.value)).group(1))
  sized = plan.L.okmi_rho_fused_workspace_bytes(basis.handle, 112, _native.PREC['bf16x6'], 1)
  assert need <= sized
  for nbytes in (need, sized):
    print('case', codes, points, nbytes, flush=True)
    plan.ws = torch.empty(-(-nbytes // 8), dtype=torch.float64, device=plan.rho.device)
    plan.rho.fill_(float('nan'))
    plan.delta.fill_(float('nan'))
    plan.launch()
    for a, b in zip(plan.result(), whole):
      assert numpy.array_equal(a, b)
