'''A call on more than 2^30 points, which no launch of one workgroup per 64
points holds: every value is written, and chosen ones are those of a call on
these points alone.
'''
import ctypes

import numpy
import pytest

pytestmark = pytest.mark.gpu
AXES = (1024, 1024, 1031)


@pytest.mark.parametrize('kind,nmo', [('ao', 1), ('mo', 1), ('rho', 65)])
def test_more_than_2_30_points(kind, nmo):
  import torch
  from orbkit_amd import _native, core
  from orbkit_amd.basis import device_basis
  from test_f64_edges import _molecule
  if torch.cuda.mem_get_info()[0] < 40 << 30:
    pytest.skip('needs 40 GB of device memory')
  print('case', kind, flush=True)
  qc = _molecule(1, 's', True, nmo)
  basis = device_basis(qc.geo_spec, qc.ao_spec)
  L = _native.lib()
  V = lambda t: ctypes.c_void_p(t.data_ptr())
  C = torch.as_tensor(qc.mo_spec.get_coeffs(), device='cuda')
  occ = torch.as_tensor(qc.mo_spec.get_occ(), device='cuda')
  code = (ctypes.c_int * 1)(0)
  ws = torch.empty(1 << 30, dtype=torch.uint8, device='cuda')

  def call(grid, out):
    n = grid.npts
    if kind == 'ao':
      rc = L.okmi_ao_eval(basis.handle, ctypes.byref(grid.desc), 0, n, code, 1, _native.OKMI_F64, V(out), n, core._stream())
    elif kind == 'mo':
      rc = L.okmi_mo_eval(basis.handle, ctypes.byref(grid.desc), 0, n, code, 1, V(C), nmo, V(out), n, V(ws), ws.numel(),
                          core._stream())
    else:
      rc = L.okmi_rho(basis.handle, ctypes.byref(grid.desc), 0, n, V(C), V(occ), nmo, None, 0, V(out), None, n, None,
                      V(ws), ws.numel(), core._stream())
    _native.check(rc, kind)
    return out
  axes = [numpy.linspace(-6, 6, n) for n in AXES]
  big = core.DeviceGrid(*axes, regular=True)
  got = call(big, torch.full((big.npts,), float('nan'), dtype=torch.float64, device='cuda'))
  assert not bool(torch.isnan(got).any())
  rng = numpy.random.default_rng(1)
  at = [numpy.concatenate([rng.integers(0, n, 500), numpy.array([0, n - 1, n // 2, n - 1])]) for n in AXES]
  few = core.DeviceGrid(*[a[i] for a, i in zip(axes, at)], regular=False)
  want = call(few, torch.empty(few.npts, dtype=torch.float64, device='cuda')).cpu().numpy()
  index = torch.as_tensor((at[0] * AXES[1] + at[1]) * AXES[2] + at[2], device='cuda')
  # (FP64, the same operations per point in either order of the points: to rounding)
  assert numpy.max(numpy.abs(got[index].cpu().numpy() - want)) <= 1e-14 * numpy.max(numpy.abs(want))
