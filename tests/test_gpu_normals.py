"""The FP64 thermal normals against Box-Muller in extended precision from the same Philox words.  Radius and cosine
or sine are each within 1.7e-16 of the exact ones and their product is rounded once (1.1e-16): 4.5e-16 in all, also
where a cosine is near zero; 5e-16 allows the extended reference its own rounding."""
import numpy as np
import pytest

import refcases as RC
from vampire_amd.context import FP64, Context

pytestmark = pytest.mark.gpu


def _philox(counter, key):
    """Philox-4x32-10 (Salmon et al., SC11) over arrays of counters."""
    c = [np.asarray(x, dtype=np.uint64) for x in counter]
    k = [np.uint64(x) for x in key]
    mask = np.uint64(0xFFFFFFFF)
    for _ in range(10):
        p0, p1 = c[0] * np.uint64(0xD2511F53), c[2] * np.uint64(0xCD9E8D57)
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ k[0], p1 & mask, (p0 >> np.uint64(32)) ^ c[3] ^ k[1], p0 & mask]
        k = [(k[0] + np.uint64(0x9E3779B9)) & mask, (k[1] + np.uint64(0xBB67AE85)) & mask]
    return c


def _turn(word):
    """(sin, cos) of 2 pi (word + 1/2) 2^-32 in extended precision, the quadrant taken out exactly."""
    q = ((word + np.uint64(1 << 29)) >> np.uint64(30)).astype(np.int64)
    t = (word.astype(np.int64) - (q << 30)).astype(np.longdouble) + np.longdouble(0.5)
    two_pi = 8 * np.arctan(np.longdouble(1))
    s, c = np.sin(two_pi * t / 2**32), np.cos(two_pi * t / 2**32)
    q &= 3
    return np.choose(q, [s, c, -s, -c]), np.choose(q, [c, -s, -c, s])


@pytest.mark.parametrize("step", [0, 5, (1 << 32) + 7])
def test_normals_match_extended_precision(gpu, step):
    n, seed = 300_001, 12345
    with Context(RC.isolated_spins(n), precision=FP64, seed=seed) as c:
        dev = c.thermal_noise(step)
    i = np.arange(n, dtype=np.uint64)
    full = lambda v: np.full(n, v, dtype=np.uint64)
    w = _philox([i, full(step & 0xFFFFFFFF), full(step >> 32), full(0)], (seed & 0xFFFFFFFF, seed >> 32))
    radius = [np.sqrt(-2 * np.log((x.astype(np.longdouble) + np.longdouble(0.5)) / 2**32)) for x in (w[0], w[2])]
    (s1, c1), (_, c2) = _turn(w[1]), _turn(w[3])
    for got, ref in zip(dev, (radius[0] * c1, radius[0] * s1, radius[1] * c2)):
        assert (np.abs(got - ref) <= 5e-16 * np.abs(ref)).all()
