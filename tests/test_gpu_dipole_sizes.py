"""The dipole field at the edges of its kernels: source cells around a pass of 256, rows that do not fill a
tile of four, empty cells, cells of one atom and of more than a workgroup's 256, a non-magnetic material,
basis-major order.  FP64 equals the oracle's sums bit for bit (same terms, same order)."""
import numpy as np
import pytest

import refcases as RC
from oracle import oracle as O
from vampire_amd import system as S
from vampire_amd.context import FP32, FP64, Context

pytestmark = pytest.mark.gpu


def _cells(n, nc, nl, seed):
    """nc cells of which nl hold atoms: one with 600 atoms (if there are as many), the rest spread."""
    rng = np.random.default_rng(seed)
    local = np.sort(rng.permutation(nc)[:nl]).astype(np.int32)
    cell = local[rng.integers(0, nl, n)]
    cell[:nl] = local                                # no local cell is empty
    cell[nl:min(n, nl + 600)] = local[0]
    return dict(num_cells=nc, local_cell=local, atom_cell=cell.astype(np.int32), volume=rng.uniform(50.0, 90.0, nc),
                tensor=rng.standard_normal((6, nl, nc)), update_rate=1)


@pytest.mark.parametrize("nc,nl", [(1, 1), (3, 2), (64, 5), (255, 254), (256, 256), (257, 9), (512, 131), (700, 698)])
def test_field_equals_the_oracle(gpu, nc, nl):
    s = RC.isolated_spins(max(2000, 3 * nl))
    sp = S.random_spins(s.n, nc)
    cells = _cells(s.n, nc, nl, nc + nl)
    o = O.Oracle(s)
    o.set_dipole(spins=sp, **cells)
    B, Hd = o.dipole_fields()[:2]
    for precision in (FP64, FP32):
        with Context(s, precision=precision, seed=1) as c:
            c.set_dipole(**cells, spins=sp)
            b, hd = c.dipole_field()
            if precision == FP64:
                assert np.array_equal(b, B) and np.array_equal(hd, Hd)
                h = c.fields()[1]                    # the atoms' own copy: H_ext without other terms
                assert np.array_equal(h, B)
            else:
                assert np.abs(hd - Hd).max() <= 1e-6 * np.abs(Hd).max()


def test_field_in_basis_major_order(gpu):
    s = S.ferromagnet("fcc", 6)
    sp = S.random_spins(s.n, 9)
    cells = _cells(s.n, 40, 37, 5)
    o = O.Oracle(s)
    o.set_dipole(spins=sp, **cells)
    B, Hd = o.dipole_fields()[:2]
    with Context(s, precision=FP64, seed=1) as c:
        assert c.atom_period > 1
        c.set_dipole(**cells, spins=sp)
        b, hd = c.dipole_field()
        assert np.array_equal(b, B) and np.array_equal(hd, Hd)
        h = c.fields()[1]
        assert np.array_equal(h, B)


def test_non_magnetic_atoms_have_no_field(gpu):
    s = S.config_c4(8, 8, 4)
    cells = _cells(s.n, 9, 9, 2)
    with Context(s, precision=FP64, seed=1) as c:
        c.set_dipole(**cells, spins=S.random_spins(s.n, 4), magnetic=[1, 0])
        b, hd = c.dipole_field()
        assert not b[:, s.type == 1].any() and not hd[:, s.type == 1].any()
        assert b[:, s.type == 0].all() and hd[:, s.type == 0].all()
        c.set_dipole(**cells, spins=S.random_spins(s.n, 4), magnetic=[0, 0])
        b, hd = c.dipole_field()
        assert not b.any() and not hd.any()
