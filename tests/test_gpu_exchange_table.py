"""Exchange tables staged in LDS (up to 8 KiB) and read from memory (beyond) give the oracle's step: tables of
each exchange type on both sides of the line, FP64 against the oracle, Heun and midpoint, in the two-kernel
step (the CSR layout walks its rows and never stages the table)."""
import numpy as np
import pytest

from oracle import oracle as O
from vampire_amd import system as S
from vampire_amd.context import FP32, FP64, Context

pytestmark = pytest.mark.gpu


def _system(exchange_type, entries):
    """A 36x36x54 SC block (70k atoms: beyond the whole-step kernel) whose bonds take `entries` values."""
    s = S.ferromagnet("sc", 36, Lz=54)
    rng = np.random.default_rng(entries)
    width = {S.ISOTROPIC: 1, S.VECTORIAL: 3, S.TENSORIAL: 9}[exchange_type]
    table = 350.0 * (1.0 + 0.2 * rng.standard_normal((entries, width)))
    iid = rng.integers(0, entries, s.nnz).astype(np.int32)
    iid[:entries] = np.arange(entries)
    return S.dataclasses.replace(s, exchange_type=exchange_type, exchange=table, nbr_iid=iid)


@pytest.mark.parametrize("exchange_type,reals", [(S.ISOTROPIC, 1), (S.VECTORIAL, 3), (S.TENSORIAL, 9)])
@pytest.mark.parametrize("kib", [1, 8, 9])
def test_tables_on_both_sides_of_the_line(gpu, exchange_type, reals, kib):
    entries = kib * 1024 // (8 * reals)
    s = _system(exchange_type, entries)
    sp = S.random_spins(s.n, 2)
    o = O.Oracle(s)
    o.set_conditions(300.0, (0.0, 0.1, 0.2))
    for integrator in ("llg_heun", "llg_midpoint"):
        ref = getattr(o, integrator)(sp, 2, seed=6)
        out = {}
        for precision in (FP64, FP32):
            with Context(s, precision=precision, seed=6, topology="ell") as c:
                c.set_conditions(300.0, (0.0, 0.1, 0.2))
                c.set_spins(sp)
                getattr(c, integrator)(2)
                out[precision] = c.get_spins()
        assert np.abs(out[FP64] - ref).max() <= 1e-12
        assert np.abs(out[FP32] - ref).max() <= 1e-5
