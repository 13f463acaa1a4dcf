"""Spins to the device and back through the chunked pinned transfer: every value returns to its place
bit for bit (FP32: the float nearest to it), at sizes on both sides of a chunk (131072 doubles), with
several workers, in basis-major order and over ragged replicas; a few statistics read in one piece."""
import numpy as np
import pytest

import refcases as RC
from vampire_amd import system as S
from vampire_amd.context import FP32, FP64, Context

pytestmark = pytest.mark.gpu


def _replicas():
    return S.concat_systems([S.ferromagnet("bcc", L, alpha=1.0) for L in (3, 5, 4)])


@pytest.mark.parametrize("precision", [FP64, FP32])
@pytest.mark.parametrize("make", [lambda: RC.isolated_spins(1), lambda: RC.isolated_spins(511),
                                  lambda: RC.isolated_spins(131071), lambda: RC.isolated_spins(131073),
                                  lambda: RC.isolated_spins(750_001), lambda: S.ferromagnet("fcc", 5), _replicas],
                         ids=["1", "511", "chunk-1", "chunk+1", "workers", "fcc", "bcc-replicas"])
def test_spins_round_trip(gpu, precision, make):
    s = make()
    rng = np.random.default_rng(s.n)
    sp = rng.uniform(-1.0, 1.0, (3, s.n))
    want = sp if precision == FP64 else sp.astype(np.float32).astype(np.float64)
    with Context(s, precision=precision, seed=1) as c:
        c.set_spins(sp)
        assert np.array_equal(c.get_spins(), want)
        c.set_spins(sp[::-1])                       # the slots in use again
        assert np.array_equal(c.get_spins(), want[::-1])
        if c.atom_period > 1:                       # stored in another order: the fields are the caller's
            h, _ = c.fields()
            with Context(s, precision=precision, seed=1, atom_order="caller") as d:
                d.set_spins(sp[::-1])
                assert np.array_equal(d.get_spins(), want[::-1]) and np.array_equal(d.fields()[0], h)


def test_reset_clears_sums_and_counter(gpu):
    s = S.ferromagnet("sc", 5)
    with Context(s, precision=FP64, seed=1) as c:
        c.set_spins(S.random_spins(s.n, 2))
        hs = [c.add_magnetization(np.arange(s.n) % k, k) for k in (1, 5, 40)]
        he = c.add_energy(np.arange(s.n) % 3, 3)
        for _ in range(2):
            c.stats_update()
        c.stats_reset()
        for cur, mean, count in [c.magnetization(h) for h in hs] + [c.energy(he)]:
            assert count == 0 and not mean.any() and cur.any()
        c.stats_update()
        for h in hs:
            cur, mean, count = c.magnetization(h)
            assert count == 1 and np.array_equal(cur, mean)
