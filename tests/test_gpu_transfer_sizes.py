"""Arrays to and from the device around the sizes where their way changes: one chunk (512 KiB), several, the
slots in use by the transfer before, and the dipole field spread over the atoms by the host (up to 262,144
atoms) or by the device."""
import numpy as np
import pytest

import refcases as RC
from vampire_amd import system as S
from vampire_amd.context import FP32, FP64, Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [FP64, FP32])
@pytest.mark.parametrize("n", [21_845, 21_846, 43_691, 65_537, 87_382, 174_763, 349_526])
def test_transfers_in_a_row(gpu, n, precision):
    s = RC.isolated_spins(n)
    rng = np.random.default_rng(n)
    with Context(s, precision=precision, seed=1) as c:
        for _ in range(4):
            sp = rng.uniform(-1.0, 1.0, (3, n))
            c.set_spins(rng.uniform(-1.0, 1.0, (3, n)))
            c.set_spins(sp)                              # into slots whose copies may still run
            want = sp if precision == FP64 else sp.astype(np.float32).astype(np.float64)
            assert np.array_equal(c.get_spins(), want)


@pytest.mark.parametrize("make", [lambda: RC.isolated_spins(262_144), lambda: RC.isolated_spins(262_145),
                                  lambda: S.ferromagnet("fcc", 40), lambda: S.ferromagnet("fcc", 41)],
                         ids=["host", "device", "host-fcc", "device-fcc"])
def test_dipole_field_read_on_both_sides_of_the_line(gpu, make):
    s = make()
    rng = np.random.default_rng(3)
    nc = 12
    cell = rng.integers(0, nc, s.n).astype(np.int32)
    args = dict(num_cells=nc, local_cell=np.arange(nc), atom_cell=cell, volume=rng.uniform(50.0, 90.0, nc),
                tensor=rng.standard_normal((6, nc, nc)), update_rate=1)
    with Context(s, precision=FP64, seed=1) as c:
        c.set_dipole(**args, spins=S.random_spins(s.n, 4))
        b, hd = c.dipole_field()
        assert np.array_equal(b, c.fields()[1])          # the atoms' own copy: H_ext without other terms
        for f in (b, hd):                                # one value a cell
            first = np.array([np.flatnonzero(cell == k)[0] for k in range(nc)])
            assert np.array_equal(f, f[:, first][:, cell]) and len(set(f[0, first])) == nc
