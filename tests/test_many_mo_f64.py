'''FP64 density of more than 64 MOs on both sides of the rule that chooses the
fused or the staged kernel (128 tiles of 64 points; groups of MOs).
'''
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('points', [500, 8128, 8129])
@pytest.mark.parametrize('drv', [None, ['y'], ['xx', 'yy', 'zz'], ['xy']])
@pytest.mark.parametrize('nmo', [192, 193, 400])
def test_both_sides(nmo, drv, points):
  '''Bar: that of every FP64 path against the oracle.'''
  from test_f64_edges import _check, _molecule
  print('case', nmo, drv, points, flush=True)
  _check(_molecule(3, 'sspdf', True, nmo), points, drv=drv)


@pytest.mark.parametrize('points', [100, 16400])
@pytest.mark.parametrize('nmo', [16, 20, 28, 44])
def test_rho_alone(nmo, points):
  '''Rho alone with C in place and from its transpose (160 AOs: by the MOs and the
  number of tiles).  Bar: that of every FP64 path against the oracle.'''
  from test_f64_edges import _check, _molecule
  print('case', nmo, points, flush=True)
  _check(_molecule(8, 'ssppdf', True, nmo), points)
