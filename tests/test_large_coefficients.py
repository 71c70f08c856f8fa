'''More than 4 GiB of MO coefficients: the FP64 kernel's transpose of C is reached
with 32-bit offsets from a group of MOs, not from its beginning.
'''
import ctypes

import numpy
import pytest

pytestmark = pytest.mark.gpu
NAO, NMO, POINTS = 24000, 22600, 8200   # (128 tiles: the fused kernel)


def test_more_than_4_gib_of_coefficients():
  import torch
  from orbkit_amd import _native, core
  from orbkit_amd.basis import device_basis
  from orbkit_amd.orbitals import AOClass
  assert 8 * NAO * NMO > 2 ** 32
  if torch.cuda.mem_get_info()[0] < 40 << 30:
    pytest.skip('needs 40 GB of device memory')
  rng = numpy.random.default_rng(4)
  geo = rng.uniform(-4, 4, (24, 3))
  ao = AOClass()
  for i in range(NAO):
    ao.append({'atom': i % len(geo), 'type': 's', 'pnum': 1,
               'coeffs': numpy.array([[numpy.exp(rng.uniform(-2, 1)), rng.uniform(0.2, 1)]])})
  ao.update()
  basis = device_basis(geo, ao)
  dg = core.DeviceGrid(*rng.uniform(-5, 5, (3, POINTS)), regular=False)
  L = _native.lib()
  V = lambda t: ctypes.c_void_p(t.data_ptr())
  gen = torch.Generator(device='cuda').manual_seed(1)
  C = torch.randn((NMO, NAO), dtype=torch.float64, device='cuda', generator=gen)
  occ = torch.rand(NMO, dtype=torch.float64, device='cuda', generator=gen)
  ws = torch.empty(8 * (NMO + 200) * (NAO + 200) + (1 << 30), dtype=torch.uint8, device='cuda')
  code = (ctypes.c_int * 1)(0)
  head = (basis.handle, ctypes.byref(dg.desc), 0, POINTS)
  new = lambda *s: torch.full(s, float('nan'), dtype=torch.float64, device='cuda')
  chi, mo, rho = new(NAO, POINTS), new(NMO, POINTS), new(POINTS)
  _native.check(L.okmi_ao_eval(*head, code, 1, _native.OKMI_F64, V(chi), POINTS, core._stream()), 'okmi_ao_eval')
  print('mo', flush=True)
  _native.check(L.okmi_mo_eval(*head, code, 1, V(C), NMO, V(mo), POINTS, V(ws), ws.numel(), core._stream()),
                'okmi_mo_eval')
  print('rho', flush=True)
  _native.check(L.okmi_rho(*head, V(C), V(occ), NMO, None, 0, V(rho), None, POINTS, None, V(ws), ws.numel(),
                           core._stream()), 'okmi_rho')
  want = C @ chi
  # sums of 24,000 terms of either sign: rounding grows to some 1e-14 of the largest value
  assert float((mo - want).abs().max() / want.abs().max()) <= 1e-12
  dens = (occ[:, None] * want * want).sum(0)
  assert float((rho - dens).abs().max() / dens.max()) <= 1e-12
