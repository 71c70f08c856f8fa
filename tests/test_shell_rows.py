'''okmi_fused_shell_rows, the work measure of the fused FP64 kernel: zero on a grid
far from every atom, all rows on a single point that every shell reaches, additive
over a grid split at a brick boundary, and below the count of whole chunks.
'''
import ctypes

import numpy
import pytest

pytestmark = pytest.mark.gpu


def test_fused_shell_rows():
  from orbkit_amd import _native, workloads
  from orbkit_amd.basis import device_basis
  qc, axes, info = workloads.make('medium', npts_side=24)
  b = device_basis(qc.geo_spec, qc.ao_spec)
  L = _native.lib()

  def rows(fn, x, y, z, *more):
    ax = [numpy.ascontiguousarray(a, dtype=numpy.float64) for a in (x, y, z)]
    out = ctypes.c_double()
    args = [v for a in ax for v in (a.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), len(a))]
    _native.check(fn(b.handle, *args, *more, ctypes.byref(out)), 'rows')
    return out.value
  x, y, z = axes
  shells = rows(L.okmi_fused_shell_rows, x, y, z)
  assert 0 < shells < rows(L.okmi_fused_live_rows, x, y, z, _native.PREC['f64'])
  assert rows(L.okmi_fused_shell_rows, x + 1e4, y, z) == 0.0
  assert rows(L.okmi_fused_shell_rows, x[:12], y, z) + rows(L.okmi_fused_shell_rows, x[12:], y, z) == shells
  # a brick as large as the molecule: every shell in reach of its box
  assert rows(L.okmi_fused_shell_rows, *[a[[0, -1]] for a in axes]) == 8 * b.nao
