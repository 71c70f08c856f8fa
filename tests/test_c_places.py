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


@pytest.mark.gpu
@pytest.mark.parametrize('nmo', [33, 36, 37, 40])
def test_general_basis_diagonal_second_derivatives(nmo):
  '''g shells, MO counts around the groups of 4 past two tiles of 16, C read in
  place (few tiles).  Bar: that of every FP64 path against the oracle.'''
  from test_f64_edges import _check, _molecule
  print('case', nmo, flush=True)
  _check(_molecule(2, 'spdfg', True, nmo), 100, drv=['xx', 'yy', 'zz'])
