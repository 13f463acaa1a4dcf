"""Constrained sweeps whose rounds sum the partials of the round before themselves, against those that leave it to
a launch (a replica with more than 512 partials in a colour: SC 82^3 has 538), and permutations made for many sweeps
ahead against one sweep's at a time.  Both orders of additions are the same, so the results equal bit for bit."""
import numpy as np
import pytest

from vampire_amd import system as S
from vampire_amd.context import FP32, FP64, Context

pytestmark = pytest.mark.gpu


def _upper(n, seed):
    """Random spins of the upper half sphere: with the moment along the constraint, pairs are accepted."""
    spins = S.random_spins(n, seed)
    spins[2] = np.abs(spins[2])
    return spins


def _run(system, spins, seed, precision, calls):
    with Context(system, precision=precision, seed=seed) as c:
        c.set_conditions(300.0, (0.0, 0.0, 0.5))
        c.set_spins(spins)
        c.mc_set_sigma(40.0)
        c.cmc_set_constraint(40.0, 30.0)
        for n in calls:
            c.cmc_sweep(n)
        return c.get_spins(), c.cmc_counts()


@pytest.mark.parametrize("precision", [FP32, FP64])
def test_folded_rounds_equal_unfolded(gpu, precision):
    sizes = [7, 12, 30, 82]
    systems = [S.ferromagnet("sc", n) for n in sizes]
    spins = [_upper(x.n, 7 + r) for r, x in enumerate(systems)]
    batch = S.concat_systems(systems)
    got, counts = _run(batch, np.concatenate(spins, axis=1), 21, precision, [3])
    off = batch.replica_offset
    for r in range(3):                               # alone: within the limit, so folded
        alone, n = _run(systems[r], spins[r], 21 + r, precision, [3])
        assert np.array_equal(got[:, off[r]:off[r + 1]], alone), sizes[r]
        assert np.array_equal(counts[r], n[0]) and counts[r].all()   # accepted and both kinds refused


@pytest.mark.parametrize("precision", [FP32, FP64])
@pytest.mark.parametrize("count", [1, 30])
def test_many_sweeps_equal_single_ones(gpu, count, precision):
    """130 sweeps in one call (three tables of permutations), in single sweeps, and in uneven calls."""
    system = S.concat_systems([S.ferromagnet("sc", 4 + r % 4) for r in range(count)])
    spins = _upper(system.n, 2)
    ref, n = _run(system, spins, 3, precision, [130])
    for calls in ([1] * 130, [64, 1, 65]):
        got, m = _run(system, spins, 3, precision, calls)
        assert np.array_equal(got, ref) and np.array_equal(m, n) and n[:, 0].all()
