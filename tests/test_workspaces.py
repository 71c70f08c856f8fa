'''Workspaces at the least size that the library asks for.'''
import ctypes

import numpy
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('nmo', [41, 48, 49, 64])
@pytest.mark.parametrize('drv', [['xx', 'yy', 'zz'], ['xx', 'xy']])
def test_least_f64_workspace(nmo, drv):
  '''okmi_rho and okmi_rho_fused in FP64 with okmi_rho_fused_workspace_bytes for
  64 points, MO counts that take two launches for the diagonal second
  derivatives.  Bar: that of every FP64 path against the oracle.'''
  import torch
  from orbkit_amd import _native, core
  from orbkit_amd.basis import device_basis
  from oracle import core_oracle
  from test_f64_edges import _molecule
  print('case', nmo, drv, flush=True)
  qc = _molecule(6, 'sspdf', True, nmo)
  xyz = numpy.random.default_rng(3).uniform(-5, 5, (3, 100))
  basis = device_basis(qc.geo_spec, qc.ao_spec)
  dg = core.DeviceGrid(*xyz, regular=False)
  L = _native.lib()
  V = lambda t: ctypes.c_void_p(t.data_ptr())
  C = torch.as_tensor(qc.mo_spec.get_coeffs(), device='cuda')
  occ = torch.as_tensor(qc.mo_spec.get_occ(), device='cuda')
  nbytes = L.okmi_rho_fused_workspace_bytes(basis.handle, nmo, _native.PREC['f64'], 64)
  ws = torch.empty(nbytes, dtype=torch.uint8, device='cuda')
  codes = core._codes(drv)
  head = (basis.handle, ctypes.byref(dg.desc), 0, dg.npts, V(C), V(occ), nmo, codes.ctypes.data_as(_native.P_int),
          len(codes))
  want = core_oracle.rho_compute(qc, *xyz, True, drv=drv)
  mos = core_oracle.rho_compute(qc, *xyz, True, calc_mo=True)
  for norms in (False, True):
    rho = torch.empty(dg.npts, dtype=torch.float64, device='cuda')
    delta = torch.empty((len(codes), dg.npts), dtype=torch.float64, device='cuda')
    nrm = torch.zeros(nmo, dtype=torch.float64, device='cuda')
    if norms:
      _native.check(L.okmi_rho(*head, V(rho), V(delta), dg.npts, V(nrm), V(ws), nbytes, core._stream()), 'okmi_rho')
      assert rel_err(nrm.cpu().numpy(), (mos ** 2).sum(axis=1)) <= 1e-12
    else:
      _native.check(L.okmi_rho_fused(*head, _native.PREC['f64'], V(rho), V(delta), dg.npts, V(ws), nbytes,
                                     core._stream()), 'okmi_rho_fused')
    assert rel_err(rho.cpu().numpy(), want[0]) <= 1e-12
    assert rel_err(delta.cpu().numpy(), want[1]) <= 1e-12


@pytest.mark.parametrize('codes', [[], [1, 2, 3]])
def test_least_many_mo_workspace(codes):
  '''More than 64 MOs in split bf16: the least workspace holds C padded to whole
  groups of 128 MOs and 128 points, one byte less is refused.'''
  import re
  import torch
  from orbkit_amd import core
  from orbkit_amd.basis import device_basis
  from orbkit_amd.fused import FusedPlan
  from test_f64_edges import _molecule
  qc = _molecule(6, 'sspdf', True, 130)
  basis = device_basis(qc.geo_spec, qc.ao_spec)
  dg = core.DeviceGrid(*numpy.random.default_rng(3).uniform(-5, 5, (3, 300)), regular=False)
  plan = FusedPlan(basis, dg, qc.mo_spec.get_coeffs(), qc.mo_spec.get_occ(), codes, 'bf16x6')
  plan.launch()
  whole = plan.result()
  plan.ws = plan.ws[:1]
  with pytest.raises(RuntimeError, match='too small') as e:
    plan.launch()
  need = int(re.search(r'need at least (\d+)', str(e.value)).group(1))
  assert need >= 6 * 256 * basis.nao + 128 * 4 * max(1, len(codes) + 1) * basis.nao
  plan.ws = torch.empty((need - 1) // 8, dtype=torch.float64, device='cuda')
  with pytest.raises(RuntimeError, match='too small'):
    plan.launch()
  plan.ws = torch.empty(-(-need // 8), dtype=torch.float64, device='cuda')
  plan.launch()
  assert all(numpy.array_equal(a, b) for a, b in zip(plan.result(), whole))
