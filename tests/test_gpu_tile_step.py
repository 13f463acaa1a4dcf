"""The whole-step kernel of small systems (one launch per step over tiles and their halos) against the
two-kernel step that larger systems take: the same spins bit for bit in FP64 and FP32, Heun and
midpoint, eager and from a graph, for every exchange type, ragged replicas, rows of unequal length, and
systems at the edges of a tile; the FP64 step of the smallest ones against the oracle."""
import numpy as np
import pytest

import refcases as RC
from oracle import oracle as O
from vampire_amd import system as S
from vampire_amd.context import FP32, FP64, Context

pytestmark = pytest.mark.gpu

TEMPS = (40.0, 300.0, 700.0)


def _make_tiles(c, spins):
    """A context makes its tiles once it has been asked for n / 128 steps."""
    c.set_spins(spins)
    c.llg_heun(c.n // 128 + 1)
    c.step = 0


def _step(s, precision, integrator, temps=(300.0,), steps=6, **kw):
    sp = S.random_spins(s.n, 5)
    with Context(s, precision=precision, seed=11, **kw) as c:
        _make_tiles(c, sp)
        for r in range(s.num_replicas):
            c.set_conditions(temps[r % len(temps)], (0.1, 0.0, 0.3), replica=r)
        c.set_spins(sp)
        if integrator == "graph":
            c.llg_heun_graph(2, steps // 2)
        else:
            (c.llg_heun if integrator == "heun" else c.llg_midpoint)(steps)
        return c.get_spins(), c.topology[0]


@pytest.mark.parametrize("precision", [FP64, FP32])
@pytest.mark.parametrize("integrator", ["heun", "graph", "midpoint"])
@pytest.mark.parametrize("crystal,sizes", [("sc", (17, 24, 30, 33)), ("bcc", (12, 22, 24)), ("fcc", (6, 15, 17))])
def test_batch_beyond_the_line_equals_replicas_alone(gpu, crystal, sizes, integrator, precision):
    """The batch has more slots than the whole-step kernel takes; each replica alone has fewer."""
    reps = [S.ferromagnet(crystal, L, alpha=1.0) for L in sizes]
    batch = S.concat_systems(reps)
    width = {"sc": 6, "bcc": 8, "fcc": 12}[crystal]
    assert batch.n * width > 400_000 and max(r.n for r in reps) * width <= 400_000
    off = batch.replica_offset
    sp = S.random_spins(batch.n, 5)
    for options in ({}, dict(recompute_euler=True, keep_external_field=True)):
        with Context(batch, precision=precision, seed=11, **options) as c:
            for r in range(len(reps)):
                c.set_conditions(TEMPS[r % 3], (0.1, 0.0, 0.3), replica=r)
            c.set_spins(sp)
            if integrator == "graph":
                c.llg_heun_graph(2, 3)
            else:
                (c.llg_heun if integrator == "heun" else c.llg_midpoint)(6)
            out = c.get_spins()
        if options and precision == FP32:
            continue                                  # the options change nothing in FP32 but a kept field
        for r, s in enumerate(reps):
            with Context(s, precision=precision, seed=11 + r) as c:
                c.set_conditions(TEMPS[r % 3], (0.1, 0.0, 0.3))
                _make_tiles(c, sp[:, off[r]:off[r + 1]])
                c.set_spins(sp[:, off[r]:off[r + 1]])
                if integrator == "graph":
                    c.llg_heun_graph(2, 3)
                else:
                    (c.llg_heun if integrator == "heun" else c.llg_midpoint)(6)
                assert np.array_equal(c.get_spins(), out[:, off[r]:off[r + 1]])


def _ragged():
    """Rows of 0 to 6 neighbours: an SC block open on every side with 40% of its sites removed."""
    keep = np.random.default_rng(8).random(11 * 12 * 13) >= 0.4
    lat = S.build_lattice("sc", 11, 12, 13, pbc=(False, False, False), keep=keep)
    mats = [S.Material(mu_s_muB=1.6, alpha=0.1, Ku=2e-24), S.Material(mu_s_muB=2.2, alpha=0.3)]
    types = (np.arange(lat.n) % 2).astype(np.int32)
    return S.make_system(lat, types, mats, [[5e-21, -1e-21], [-1e-21, 4e-21]], uniaxial=True)


SYSTEMS = {"1": lambda: RC.isolated_spins(1), "127": lambda: RC.isolated_spins(127), "128": lambda: RC.isolated_spins(128),
           "129": lambda: RC.isolated_spins(129), "12289": lambda: RC.isolated_spins(12289),
           "40001": lambda: RC.isolated_spins(40001), "sc2": lambda: S.ferromagnet("sc", 2),
           "fcc2": lambda: S.ferromagnet("fcc", 2), "ragged": _ragged, "film": lambda: S.config_c4(12, 10, 4),
           "vectorial": lambda: RC.system_of("film_vectorial"), "dmi": lambda: RC.system_of("film_dmi")}


@pytest.mark.parametrize("integrator", ["heun", "midpoint"])
@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_edges_against_two_kernels_and_the_oracle(gpu, name, integrator):
    """The CSR layout keeps the two-kernel step at every size."""
    s = SYSTEMS[name]()
    two, layout = _step(s, FP64, integrator, topology="csr")
    assert layout == "csr"
    one, layout = _step(s, FP64, integrator)
    assert layout != "csr" and np.array_equal(one, two)
    o = O.Oracle(s)
    o.set_conditions(300.0, (0.1, 0.0, 0.3))
    run = o.llg_heun if integrator == "heun" else o.llg_midpoint
    ref = run(S.random_spins(s.n, 5), 6, seed=11)
    assert np.abs(one - ref).max() <= 1e-12


def test_tiles_made_between_graph_replays(gpu):
    """A graph recorded from the two kernels gives way to one of the whole step when the tiles are made:
    replay by replay the same spins as eager steps."""
    s = S.ferromagnet("sc", 13)                     # 2197 atoms: tiles from the 17th step on
    sp = S.random_spins(s.n, 3)
    with Context(s, precision=FP64, seed=4) as c, Context(s, precision=FP64, seed=4, topology="csr") as d:
        for x in (c, d):
            x.set_conditions(250.0)
            x.set_spins(sp)
        for _ in range(5):
            c.llg_heun_graph(4, 2)
            d.llg_heun(8)
            assert np.array_equal(c.get_spins(), d.get_spins())
