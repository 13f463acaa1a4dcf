"""The one-launch statistics at the edges of their launches: one workgroup and several, 65,536 atoms on either
side, masks of 1 to 2048 bins (registers, LDS histograms, empty bins), every workgroup size of the block table,
rows of each layout, and batches; repeated updates, with spins changed between.  Against the oracle: relative
1e-12 of the largest value of a kind (sums of up to 72,000 doubles)."""
import numpy as np
import pytest

import refcases as RC
from oracle import oracle as O
from vampire_amd import system as S
from vampire_amd.context import FP32, FP64, Context

pytestmark = pytest.mark.gpu


def _check(s, nbins, precision=FP64, updates=2, **kw):
    rng = np.random.default_rng(s.n + nbins)
    mask = rng.integers(0, nbins, s.n).astype(np.int32)
    if nbins > 2:
        mask[mask == 1] = 0                          # an empty bin
    o = O.Oracle(s)
    o.set_conditions(100.0, (0.2, 0.1, 0.5))
    sums = [0.0, 0.0]
    with Context(s, precision=precision, seed=1, **kw) as c:
        c.set_conditions(100.0, (0.2, 0.1, 0.5))
        hm, he = c.add_magnetization(mask, nbins), c.add_energy(mask, nbins)
        for u in range(updates):
            sp = S.random_spins(s.n, u)
            if precision == FP32:
                sp = sp.astype(np.float32).astype(np.float64)
            c.set_spins(sp)
            c.stats_update()
            m, m_sum, mc = c.magnetization(hm)
            e, e_sum, ec = c.energy(he)
            rm, re = o.magnetization(sp, mask, nbins), o.energy(sp, mask, nbins)
            tol = 1e-12 if precision == FP64 else 1e-5
            assert mc == ec == u + 1
            assert np.abs(m - rm).max() <= 1e-12 * max(1.0, np.abs(rm).max())
            assert np.abs(e - np.reshape(re, e.shape)).max() <= tol * np.abs(re).max()
            sums = [sums[0] + m, sums[1] + e]
        assert np.allclose(m_sum, sums[0], rtol=1e-14, atol=1e-14)
        assert np.allclose(e_sum[:, :max(nbins - 1, 0)], sums[1][:, :max(nbins - 1, 0)], rtol=1e-14, atol=1e-12)


@pytest.mark.parametrize("n", [1, 63, 256, 257, 4097, 65536, 65537, 72001])
def test_sizes(gpu, n):
    _check(RC.isolated_spins(n), 2)


@pytest.mark.parametrize("nbins", [1, 2, 4, 5, 8, 9, 16, 17, 300, 2048])
def test_bins(gpu, nbins):
    _check(S.ferromagnet("fcc", 7), nbins)


@pytest.mark.parametrize("block", [64, 192, 512])
@pytest.mark.parametrize("topology", ["csr", "ell", "stencil"])
def test_layouts(gpu, block, topology):
    for precision in (FP64, FP32):
        _check(S.ferromagnet("bcc", 9), 3, precision, block_size=block, topology=topology)


def test_film_and_batch(gpu):
    _check(S.config_c4(40, 30, 5), 3)
    reps = [S.ferromagnet("sc", L) for L in (5, 12, 9)]
    batch = S.concat_systems(reps)
    off = batch.replica_offset
    sp = S.random_spins(batch.n, 3)
    mask = np.repeat(np.arange(3), np.diff(off)).astype(np.int32)
    with Context(batch, precision=FP64, seed=1) as c:
        he = c.add_energy(mask, 4)
        for r in range(3):
            c.set_conditions(50.0, (0.0, 0.0, 0.1 * (r + 1)), replica=r)
        c.set_spins(sp)
        c.stats_update()
        e = c.energy(he)[0]
    for r, s in enumerate(reps):
        o = O.Oracle(s)
        o.set_conditions(50.0, (0.0, 0.0, 0.1 * (r + 1)))
        ref = np.reshape(o.energy(sp[:, off[r]:off[r + 1]], np.zeros(s.n, np.int32), 2), (5, 2))[:, 0]
        assert np.abs(e[:, r] - ref).max() <= 1e-12 * np.abs(ref).max()
