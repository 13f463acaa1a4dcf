"""An energy statistic does not depend on the launch shape of the step kernels: contexts of one system that
differ in workgroup size, or have been autotuned, add the same terms in the same order, bit for bit."""
import numpy as np
import pytest

from vampire_amd import system as S
from vampire_amd.context import FP32, FP64, Context

pytestmark = pytest.mark.gpu

SYSTEMS = {"sc30": lambda: S.ferromagnet("sc", 30), "fcc27": lambda: S.ferromagnet("fcc", 27),
           "film": lambda: S.config_c4(70, 70, 6),
           "batch": lambda: S.concat_systems([S.ferromagnet("bcc", L) for L in (9, 20, 13)])}


@pytest.mark.parametrize("precision", [FP64, FP32])
@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_energies_are_the_same_for_every_workgroup_size(gpu, name, precision):
    s = SYSTEMS[name]()
    sp = S.random_spins(s.n, 4)
    out = []
    for block, tune in ((256, False), (64, False), (128, False), (192, False), (512, False), (64, True)):
        with Context(s, precision=precision, seed=1, block_size=block) as c:
            c.set_conditions(300.0, (0.1, 0.0, 0.4))
            c.set_spins(sp)
            if tune:
                c.autotune(4)
            hs = [c.add_energy(np.zeros(s.n, np.int32), 2), c.add_energy((np.arange(s.n) % 3).astype(np.int32), 4)]
            c.stats_update()
            out.append([c.energy(h)[0] for h in hs])
    for other in out[1:]:
        for a, b in zip(out[0], other):
            assert a.any() and np.array_equal(a, b)
