'''FP64 kernel on bases whose shells have several general row maps (row factors as
in ORCA output): shells with the same map are taken together, the others apart.
'''
import numpy
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('nmo', [3, 20, 66])
@pytest.mark.parametrize('drv', [None, ['x', 'y', 'z'], ['xx', 'yy', 'zz'], ['xy', 'zz']])
@pytest.mark.parametrize('spherical', [True, False])
@pytest.mark.parametrize('kinds', [1, 2, None])
def test_row_factors(kinds, spherical, drv, nmo):
  '''kinds: different sets of row factors, dealt to the shells of a type in turn
  (None: each shell its own).  Bar: that of every FP64 path against the oracle.'''
  from test_f64_edges import _check, _molecule
  print('case', kinds, spherical, drv, nmo, flush=True)
  qc = _molecule(5, 'spdfg', spherical, nmo)
  rng = numpy.random.default_rng(8)
  sets = rng.uniform(0.5, 2.0, (kinds or 1000, 15))
  rows = []
  for i, c in enumerate(qc.ao_spec.get_nlxlylz_per_cont()):
    rows.append(sets[i // 5 % kinds if kinds else i][:c])
  qc.ao_spec[0]['N'] = numpy.concatenate(rows)[:, numpy.newaxis]
  _check(qc, 300, drv=drv)
  if drv is None or drv == ['xy', 'zz']:
    _check(qc, 300, drv=drv, calc_mo=True)
