"""Conditions carried by the next step's launch against conditions written to the device table at once (a
context that evaluates its fields after every change): the same spins and statistics bit for bit, whatever
call comes next, for tables that a launch carries (192 bytes) and larger ones."""
import numpy as np
import pytest

from vampire_amd import system as S
from vampire_amd.context import FP32, FP64, FUSED, PLAIN, Context

pytestmark = pytest.mark.gpu


def _alloy(L):
    lat = S.build_lattice("sc", L, L, L)
    mats = [S.Material(mu_s_muB=1.6, alpha=0.2, Ku=2e-24, applied_field_strength=0.5), S.Material(mu_s_muB=2.2, alpha=0.3)]
    return S.make_system(lat, (np.arange(lat.n) % 2).astype(np.int32), mats, [[5e-21, -1e-21], [-1e-21, 4e-21]],
                         uniaxial=True)


SYSTEMS = {"one": lambda: S.ferromagnet("sc", 6), "alloy": lambda: _alloy(6),
           "batch4": lambda: S.concat_systems([S.ferromagnet("sc", L) for L in (3, 4, 5, 6)]),
           "batch5": lambda: S.concat_systems([S.ferromagnet("sc", L) for L in (3, 4, 5, 6, 4)]),
           "alloys": lambda: S.concat_systems([_alloy(4), _alloy(6)]),
           "large": lambda: S.ferromagnet("sc", 42)}        # the two-kernel step


def _run(s, precision, kernel, at_once):
    rng = np.random.default_rng(1)
    out = []
    with Context(s, precision=precision, kernel=kernel, seed=3) as c:
        c.set_spins(S.random_spins(s.n, 2))
        he = c.add_energy(s.type, len(s.materials) + 1)
        c.cmc_set_constraint(30.0, 10.0)

        def change():
            for r in range(s.num_replicas):
                c.set_conditions(float(rng.uniform(10.0, 600.0)), rng.uniform(-1.0, 1.0, 3), local_applied=True, replica=r)
            if at_once:
                c.fields()

        def energies():
            c.stats_update()
            out.append(c.energy(he)[0])

        graph = (lambda: c.llg_heun_graph(2, 1)) if kernel == FUSED else (lambda: c.llg_heun(2))
        for call in (lambda: c.llg_heun(1), lambda: c.llg_heun(2), lambda: c.llg_midpoint(1), energies, graph,
                     lambda: c.mc_sweep(1), lambda: c.mc_sweep(5), lambda: c.cmc_sweep(1), lambda: c.llg_heun(1)):
            change()
            call()
            out.append(c.get_spins())
            change()
            change()
            if not at_once:
                c.set_demag_field((0.0, 0.0, 0.01))
                c.set_demag_field((0.0, 0.0, 0.0))
            call()
            energies()
            out.append(c.get_spins())
    return out


@pytest.mark.parametrize("kernel", [FUSED, PLAIN])
@pytest.mark.parametrize("precision", [FP64, FP32])
@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_carried_conditions_equal_written_ones(gpu, name, precision, kernel):
    s = SYSTEMS[name]()
    for a, b in zip(_run(s, precision, kernel, False), _run(s, precision, kernel, True)):
        assert np.array_equal(a, b)
