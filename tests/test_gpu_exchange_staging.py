"""Exchange tables staged in words of the pass (one round of the workgroup) and in 16-byte words (more): sizes
around the line and around whole 16-byte words, workgroups of 64 to 512.  The CSR layout reads the table itself:
FP64 bit for bit; FP32 within 2e-6 after two steps (rounding of the sums, which the compiler fuses its own way)."""
import numpy as np
import pytest

from vampire_amd import system as S
from vampire_amd.context import FP32, FP64, Context

pytestmark = pytest.mark.gpu


def _system(exchange_type, entries):
    s = S.ferromagnet("sc", 15)                      # 3375 atoms
    rng = np.random.default_rng(entries)
    width = {S.ISOTROPIC: 1, S.VECTORIAL: 3, S.TENSORIAL: 9}[exchange_type]
    table = 350.0 * (1.0 + 0.2 * rng.standard_normal((entries, width)))
    iid = rng.integers(0, entries, s.nnz).astype(np.int32)
    iid[:entries] = np.arange(entries)
    return S.dataclasses.replace(s, exchange_type=exchange_type, exchange=table, nbr_iid=iid)


@pytest.mark.parametrize("block", [64, 128, 256, 512])
@pytest.mark.parametrize("exchange_type,entries", [(S.ISOTROPIC, k) for k in (2, 3, 65, 97, 98, 99, 226, 227, 482, 483, 1023, 1024)]
                         + [(S.VECTORIAL, k) for k in (2, 33, 75, 161, 341)] + [(S.TENSORIAL, k) for k in (2, 7, 25, 54, 113)])
def test_staged_table_equals_the_table_in_memory(gpu, exchange_type, entries, block):
    s = _system(exchange_type, entries)
    sp = S.random_spins(s.n, 2)
    for precision in (FP64, FP32):
        for integrator in ("llg_heun", "llg_midpoint"):
            out = []
            for topology in ("csr", "ell"):
                with Context(s, precision=precision, seed=6, topology=topology, block_size=block) as c:
                    c.set_whole_step(False)
                    c.set_conditions(300.0, (0.0, 0.1, 0.2))
                    c.set_spins(sp)
                    getattr(c, integrator)(2)
                    out.append(c.get_spins())
            if precision == FP64:
                assert np.array_equal(out[0], out[1])
            else:
                assert np.abs(out[0] - out[1]).max() <= 2e-6
