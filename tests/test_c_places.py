'''Which MO coefficients the FP64 fused kernel's lanes read (csrc/c_place.h,
compiled here for the host), walked against the bounds of C: read where the caller
has it (no padding after its last MO or row) and as the padded transpose.
'''
import itertools
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r'''
#include <cstdio>
#include <initializer_list>
#include "c_place.h"
using namespace okmi_fused;
int main()
{
    // u pass standard units, then per lane the last tile's and the last group's MO
    for (int standard = 0; standard < 2; ++standard)
        for (int pass = 0; pass < 5; ++pass)
            for (int nmo = 1; nmo <= (pass == 4 ? 40 : 64); ++nmo) {
                const int U = f64_units((nmo + 3) / 4, pass, standard, false), NT = U / 4, NR = U % 4;
                for (int ct = 0; ct < 2; ++ct) {
                    const int last = (ct ? 4 * U : nmo) - 1;
                    std::printf("mo %d %d %d %d %d", standard, pass, nmo, ct, U);
                    for (int n = 0; n < 16; ++n) std::printf(" %d", NT && !NR ? last_tile_mo(n, last, NT) : n);
                    for (int n = 0; n < 4; ++n) std::printf(" %d", NR ? last_group_mo(n, last, NT, NR) : n);
                    std::printf("\n");
                }
            }
    // l rows W R, then the row of each place
    for (int l = 1; l <= 4; ++l)
        for (int N : {2 * l + 1, (l + 1) * (l + 2) / 2})
            for (int R = 0; R < N; ++R) {
                std::printf("row %d %d 2 %d", l, N, R);
                for (int w = 0; w < 2; ++w) std::printf(" %d", split_row<2>(R, w, N));
                std::printf("\nrow %d %d 4 %d", l, N, R);
                for (int w = 0; w < 4; ++w) std::printf(" %d", split_row<4>(R, w, N));
                std::printf("\n");
            }
}
'''


@pytest.fixture(scope='module')
def lines(tmp_path_factory):
  d = tmp_path_factory.mktemp('places')
  (d / 'driver.cpp').write_text(DRIVER)
  subprocess.run(['g++', '-std=c++17', '-D__host__=', '-D__device__=', '-I', os.path.join(ROOT, 'orbkit_amd', 'csrc'),
                  str(d / 'driver.cpp'), '-o', str(d / 'driver')], check=True)
  out = subprocess.run([str(d / 'driver')], check=True, capture_output=True, text=True).stdout
  return [l.split() for l in out.splitlines()]


def test_mo_places(lines):
  '''Every place of an MO reads that MO, every place past the last one an MO
  of the launch (its occupation is zero).'''
  seen = set()
  for l in lines:
    if l[0] != 'mo':
      continue
    standard, pas, nmo, ct, U = (int(x) for x in l[1:6])
    tile, group = [int(x) for x in l[6:22]], [int(x) for x in l[22:26]]
    NT, NR = U // 4, U % 4
    have = 4 * U if ct else nmo
    read = []   # MO of each place, in order
    for j in range(NT):
      read += [16 * j + (tile[n] if NR == 0 and j == NT - 1 else n) for n in range(16)]
    for j in range(NR):
      read += [16 * NT + 4 * j + (group[n] if j == NR - 1 else n) for n in range(4)]
    assert len(read) == 4 * U >= nmo
    assert all(0 <= m < have for m in read), (standard, pas, nmo, ct, U, read)
    assert read[:nmo] == list(range(nmo))
    seen.add((standard, pas, nmo, ct))
  want = {(s, p, n, c) for s, p, c in itertools.product((0, 1), range(5), (0, 1))
          for n in range(1, 41 if p == 4 else 65)}
  assert seen == want


def test_row_places(lines):
  '''Rows of a shell spread over lane groups: every place of a row reads that
  row, every place past the last one a row of the shell.'''
  n = 0
  for l in lines:
    if l[0] == 'row':
      N, W, R = int(l[2]), int(l[3]), int(l[4])
      rows = [int(x) for x in l[5:]]
      assert len(rows) == W and all(0 <= r < N for r in rows), l
      assert rows[:N - R] == list(range(R, min(R + W, N))), l
      n += 1
  assert n == 2 * sum(2 * l + 1 + (l + 1) * (l + 2) // 2 for l in range(1, 5))


@pytest.mark.gpu
@pytest.mark.parametrize('nmo', [33, 36, 37, 40])
def test_general_basis_diagonal_second_derivatives(nmo):
  '''g shells, MO counts around the groups of 4 past two tiles of 16, C read in
  place (few tiles).  Bar: that of every FP64 path against the oracle.'''
  from test_f64_edges import _check, _molecule
  print('case', nmo, flush=True)
  _check(_molecule(2, 'spdfg', True, nmo), 100, drv=['xx', 'yy', 'zz'])


@pytest.mark.gpu
@pytest.mark.parametrize('axes', [(4, 5, 6), (33, 32, 32)])   # C in place; its transpose (512 tiles and more)
@pytest.mark.parametrize('spherical', [True, False])
def test_p_shell_at_the_end(spherical, axes):
  '''The basis ends with its only p shell, what follows C in memory is NaN, and
  so is the workspace before the call: none of it reaches the density or the MO
  values.  Bar: that of every FP64 path against the oracle.'''
  import ctypes
  import numpy
  import torch
  from conftest import rel_err
  from orbkit_amd import _native, core
  from orbkit_amd.basis import device_basis
  from oracle import core_oracle
  from test_f64_edges import _molecule
  print('case', spherical, axes, flush=True)
  qc = _molecule(1, 'sdp', spherical, 7)
  xyz = [numpy.linspace(-4, 4, n) for n in axes]
  basis = device_basis(qc.geo_spec, qc.ao_spec)
  dg = core.DeviceGrid(*xyz, regular=True)
  L, nan = _native.lib(), float('nan')
  C = qc.mo_spec.get_coeffs()
  held = torch.full((C.size + 512,), nan, dtype=torch.float64, device='cuda')
  held[:C.size] = torch.as_tensor(C.reshape(-1), device='cuda')
  occ = torch.as_tensor(qc.mo_spec.get_occ(), device='cuda')
  ws = torch.empty(L.okmi_workspace_bytes(basis.handle, 7, dg.npts) // 8 + 1, dtype=torch.float64, device='cuda')
  V = lambda t: ctypes.c_void_p(t.data_ptr())
  codes = numpy.arange(4, dtype=numpy.intc)
  P = lambda a: a.ctypes.data_as(_native.P_int)
  for drv in ([], [1, 2, 3], [4, 5, 6]):
    d = numpy.array(drv, dtype=numpy.intc)
    rho = torch.empty(dg.npts, dtype=torch.float64, device='cuda')
    delta = torch.empty((max(1, len(d)), dg.npts), dtype=torch.float64, device='cuda')
    ws.fill_(nan)
    _native.check(L.okmi_rho(basis.handle, ctypes.byref(dg.desc), 0, dg.npts, V(held), V(occ), len(C), P(d), len(d),
                             V(rho), V(delta), dg.npts, None, V(ws), ws.numel() * 8, core._stream()), 'okmi_rho')
    want = core_oracle.rho_compute(qc, *xyz, False, drv=[['x', 'y', 'z', 'xx', 'yy', 'zz'][k - 1] for k in drv] or None)
    want = want if drv else (want,)
    assert rel_err(rho.cpu().numpy(), want[0].reshape(-1)) <= 1e-12
    if drv:
      assert rel_err(delta.cpu().numpy(), want[1].reshape(len(drv), -1)) <= 1e-12
  mo = torch.empty((4, len(C), dg.npts), dtype=torch.float64, device='cuda')
  ws.fill_(nan)
  _native.check(L.okmi_mo_eval(basis.handle, ctypes.byref(dg.desc), 0, dg.npts, P(codes), 4, V(held), len(C), V(mo),
                               dg.npts, V(ws), ws.numel() * 8, core._stream()), 'okmi_mo_eval')
  want = core_oracle.rho_compute(qc, *xyz, False, calc_mo=True, drv=[None, 'x', 'y', 'z'])
  assert rel_err(mo.cpu().numpy(), want.reshape(4, len(C), -1)) <= 1e-12
