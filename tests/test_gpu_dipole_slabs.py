"""A dipole tensor larger than the 32 MiB that are laid out at a time: several slabs of rows, the last one
ragged (1303 = 4 x 325 + 3).  FP64 equals the oracle's sums bit for bit (same terms, same order)."""
import numpy as np
import pytest

import refcases as RC
from oracle import oracle as O
from vampire_amd import system as S
from vampire_amd.context import FP64, Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc,nl", [(1303, 1303), (1500, 1301), (2000, 700)])
def test_field_of_several_slabs_equals_the_oracle(gpu, nc, nl):
    rng = np.random.default_rng(nc + nl)
    s = RC.isolated_spins(3 * nc)
    sp = S.random_spins(s.n, nc)
    local = np.sort(rng.permutation(nc)[:nl]).astype(np.int32)
    cell = local[rng.integers(0, nl, s.n)]
    cell[:nl] = local                                # no local cell is empty
    cells = dict(num_cells=nc, local_cell=local, atom_cell=cell.astype(np.int32), volume=rng.uniform(50.0, 90.0, nc),
                 tensor=rng.standard_normal((6, nl, nc)), update_rate=1)
    assert cells["tensor"].nbytes > 32 << 20
    o = O.Oracle(s)
    o.set_dipole(spins=sp, **cells)
    B, Hd = o.dipole_fields()[:2]
    with Context(s, precision=FP64, seed=1) as c:
        c.set_dipole(**cells, spins=sp)
        b, hd = c.dipole_field()
        assert np.array_equal(b, B) and np.array_equal(hd, Hd)
