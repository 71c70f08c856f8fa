'''FP32 densities with four MO tiles (49 to 64 MOs), whose AO rows come from the
Cartesian values: every row map, against the FP64 path.  Bar 2.5e-7 norm-wise:
AO values and C rounded to FP32 (6e-8 each) and FP32 sums.
'''
import numpy
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('points', [None, 129])
@pytest.mark.parametrize('nmo', [49, 64])
def test_f32_four_tiles(nmo, points):
  import torch
  if not torch.cuda.is_available():
    pytest.skip('no HIP device')
  from orbkit_amd import core, workloads
  from orbkit_amd.basis import device_basis
  from orbkit_amd.core import DeviceGrid
  from orbkit_amd.fused import rho_fused
  qc, axes, _ = workloads.make('medium', npts_side=14, nmo=64)
  basis = device_basis(qc.geo_spec, qc.ao_spec)
  C, occ = qc.mo_spec.get_coeffs()[:nmo], numpy.full(nmo, 2.0)
  rng = numpy.random.default_rng(4)
  g = DeviceGrid(*axes, regular=True) if points is None else DeviceGrid(
      *[rng.uniform(a[0] + 4, a[-1] - 4, points) for a in axes], regular=False)
  print('case', nmo, points, flush=True)
  got, want = rho_fused(basis, g, C, occ, [], 'f32')[0], core.eval_rho(basis, g, C, occ, [])[0]
  assert numpy.linalg.norm(got - want) <= 2.5e-7 * numpy.linalg.norm(want)
