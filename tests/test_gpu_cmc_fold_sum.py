"""A constrained sweep whose first round adds the full sum's partials itself (up to 8192 a replica) against one
that leaves them to a launch: in workgroups of 64 atoms FCC 52^3 has 8788 partials, so a batch that holds it takes
the launch, and its smaller replicas alone do not.  The order of additions is the same: equal bit for bit."""
import numpy as np
import pytest

from vampire_amd import system as S
from vampire_amd.context import FP32, FP64, Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [FP32, FP64])
def test_first_round_on_both_sides_of_the_line(gpu, precision):
    systems = [S.ferromagnet("fcc", n) for n in (10, 20, 52)]
    spins = []
    for r, x in enumerate(systems):
        sp = S.random_spins(x.n, 3 + r)
        sp[2] = np.abs(sp[2])                        # with the moment along the constraint, pairs are accepted
        spins.append(sp)

    def run(system, sp, seed):
        with Context(system, precision=precision, seed=seed, block_size=64) as c:
            c.set_conditions(300.0, (0.0, 0.0, 0.5))
            c.set_spins(sp)
            c.cmc_set_constraint(40.0, 30.0)
            c.cmc_sweep(4)
            return c.get_spins(), c.cmc_counts()

    batch = S.concat_systems(systems)
    got, counts = run(batch, np.concatenate(spins, axis=1), 21)
    off = batch.replica_offset
    for r in range(3):
        alone, n = run(systems[r], spins[r], 21 + r)
        assert np.array_equal(got[:, off[r]:off[r + 1]], alone) and np.array_equal(counts[r], n[0]) and counts[r].all()
