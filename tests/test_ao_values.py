'''AO values in memory at the edges of the 64-point tiles, which the card's dies take
in eighths: every column of every row is written, and nothing past the last point.
Both value types.
'''
import ctypes

import numpy
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', ['F64', 'F32'])
@pytest.mark.parametrize('drv', [None, ['x', 'y', 'z'], ['xx', 'yy', 'zz'], ['yz', 'x']])
@pytest.mark.parametrize('npts', [1, 64, 65, 7 * 64, 9 * 64 - 1, 15 * 64 + 1, 16 * 64, 9999])
@pytest.mark.parametrize('spherical', [True, False])
def test_every_tile(spherical, npts, drv, dtype):
  '''Bars: that of every FP64 path against the oracle; for FP32, its rounding (6e-8)
  and an exponential to 2.6e-9, whose share cancelling terms enlarge: 2e-7.'''
  import torch
  if not torch.cuda.is_available():
    pytest.skip('no HIP device')
  from orbkit_amd import _native, core
  from orbkit_amd.basis import device_basis
  from oracle import core_oracle
  from test_f64_edges import _molecule
  print('case', spherical, npts, drv, dtype, flush=True)
  qc = _molecule(3, 'spdfg', spherical, 1)
  points = numpy.random.default_rng(2).uniform(-5, 5, (3, npts))
  grid = core.DeviceGrid(*points, regular=False)
  basis = device_basis(qc.geo_spec, qc.ao_spec)
  codes = core._codes(drv or [None])
  ld = npts + 3
  out = torch.full((len(codes), basis.nao, ld), float('nan'), device='cuda',
                   dtype=torch.float64 if dtype == 'F64' else torch.float32)
  _native.check(_native.lib().okmi_ao_eval(basis.handle, ctypes.byref(grid.desc), 0, npts,
                                           codes.ctypes.data_as(_native.P_int), len(codes), getattr(_native, 'OKMI_' + dtype),
                                           ctypes.c_void_p(out.data_ptr()), ld, core._stream()), 'okmi_ao_eval')
  got = out.cpu().numpy()
  assert numpy.isnan(got[..., npts:]).all()
  for j, d in enumerate(drv or [None]):
    want = core_oracle.rho_compute(qc, *points, True, calc_ao=True, drv=d and [d])
    want = want.reshape(basis.nao, npts)
    assert abs(got[j, :, :npts] - want).max() <= (1e-12 if dtype == 'F64' else 2e-7) * abs(want).max()
