"""Both forms of a small system's step against the references: the parity tests of the Heun and midpoint
integrators once more with the two kernels kept (set_whole_step(False)), where larger systems and small ones
alike run k_fused_* and k_mid_* over ELL and stencil rows of every exchange type with what the options keep or
recompute; and once with the whole-step kernel known to be in use.  Then both forms side by side, bit for bit."""
import numpy as np
import pytest

import refcases as RC
import test_gpu_llg as LLG
import test_gpu_midpoint as MID
from vampire_amd import system as S
from vampire_amd.context import FP32, FP64, FUSED, PLAIN, Context

pytestmark = pytest.mark.gpu


class TwoKernels(Context):
    def __init__(self, *args, **kw):
        super().__init__(*args, **kw)
        self.set_whole_step(False)

    def close(self):
        if getattr(self, "h", None):
            assert self.tiles == 0
        super().close()


class WholeStep(Context):
    """A context that has taken the steps after which it makes its tiles, and is as it was before them."""

    def __init__(self, *args, **kw):
        super().__init__(*args, **kw)
        self.set_conditions(0.0)
        self.set_spins(S.random_spins(self.n, 99))
        self.llg_heun(self.n // 128 + 1)
        assert self.tiles > 0
        self.set_spins(np.zeros((3, self.n)))
        self.step = 0


@pytest.fixture(params=[TwoKernels, WholeStep], ids=["two-kernels", "whole-step"])
def form(request, monkeypatch):
    for module in (LLG, MID):
        monkeypatch.setattr(module, "Context", request.param)
    return request.param


ROWS = ["ell", "stencil"]
FUSED_KERNELS = [k for k in LLG.KERNELS if k != PLAIN]


@pytest.mark.parametrize("topology", ROWS)
@pytest.mark.parametrize("kernel", FUSED_KERNELS)
@pytest.mark.parametrize("name", LLG.GOLDEN_CASES)
def test_trajectory(gpu, form, name, kernel, topology):
    LLG.test_trajectory_matches_reference(gpu, name, kernel, topology)


@pytest.mark.parametrize("kernel", FUSED_KERNELS)
def test_c0(gpu, form, kernel):
    LLG.test_c0_1000_steps_philox(gpu, kernel)


def test_c0_golden(gpu, form):
    LLG.test_c0_golden_1000_steps(gpu)


@pytest.mark.parametrize("name", LLG.GOLDEN_CASES)
def test_fp32(gpu, form, name):
    LLG.test_fp32_matches_reference_same_normals(gpu, name, FUSED)


@pytest.mark.parametrize("kernel", FUSED_KERNELS)
def test_demag(gpu, form, kernel):
    LLG.test_thin_film_demag_matches_reference(gpu, kernel)


@pytest.mark.parametrize("kernel", FUSED_KERNELS)
@pytest.mark.parametrize("dims,lds", [((16, 16, 4), True), ((24, 24, 6), False)])
def test_ragged_stencils(gpu, form, dims, lds, kernel):
    LLG.test_ragged_stencils_small_and_large_tables(gpu, dims, lds, kernel)


def test_graphs_and_replicas(gpu, form):
    LLG.test_graph_equals_eager(gpu)
    LLG.test_eager_and_graph_interleaved_equal_eager(gpu)
    LLG.test_replicas_equal_standalone(gpu)


@pytest.mark.parametrize("keep", [False, True])
@pytest.mark.parametrize("topology", ROWS)
@pytest.mark.parametrize("name", MID.MID_CASES)
def test_midpoint_trajectory(gpu, form, name, topology, keep):
    MID.test_midpoint_matches_reference(gpu, name, topology, keep)


def test_midpoint_philox(gpu, form):
    MID.test_midpoint_philox_matches_oracle(gpu)


@pytest.mark.parametrize("precision", [FP64, FP32])
@pytest.mark.parametrize("integrator", ["heun", "graph", "midpoint"])
@pytest.mark.parametrize("name", LLG.GOLDEN_CASES)
def test_forms_equal_bit_for_bit(gpu, name, integrator, precision):
    f, s = RC.load(name), RC.system_of(name)
    T, H = RC.conditions(name)
    out = []
    for make in (TwoKernels, WholeStep):
        with make(s, precision=precision, seed=5) as c:
            c.set_conditions(T, H, **RC.flags(name))
            c.set_spins(f["spins_in"])
            if integrator == "graph":
                c.llg_heun_graph(4, 3)
            else:
                (c.llg_heun if integrator == "heun" else c.llg_midpoint)(12)
            out.append(c.get_spins())
    assert np.array_equal(out[0], out[1])


def test_switching_between_forms_drops_the_recorded_graph(gpu):
    s = S.ferromagnet("fcc", 6)
    sp = S.random_spins(s.n, 8)
    with WholeStep(s, precision=FP32, seed=2) as c, TwoKernels(s, precision=FP32, seed=2) as d:
        for x in (c, d):
            x.set_conditions(300.0)
            x.set_spins(sp)
        for on in (True, False, False, True):
            c.set_whole_step(on)
            assert (c.tiles > 0) == on
            c.llg_heun_graph(4, 2)
            d.llg_heun(8)
            assert np.array_equal(c.get_spins(), d.get_spins())


@pytest.mark.parametrize("precision", [FP64, FP32])
@pytest.mark.parametrize("before", [0, 40])
def test_autotuning_leaves_the_run_as_it_was(gpu, precision, before):
    """Before and after the tiles are made: spins, step counter and form stay, later steps give the same spins."""
    s = S.ferromagnet("bcc", 13)                     # 4394 atoms: tiles from the 34th step on
    sp = S.random_spins(s.n, 6)
    with Context(s, precision=precision, seed=3) as c, TwoKernels(s, precision=precision, seed=3) as d:
        for x in (c, d):
            x.set_conditions(200.0, (0.0, 0.1, 0.2))
            x.set_spins(sp)
            x.llg_heun(before)
        tiles = c.tiles
        assert c.autotune(12) in (64, 128, 256, 512)
        assert c.tiles == tiles and c.step == before and np.array_equal(c.get_spins(), d.get_spins())
        for x in (c, d):
            x.llg_heun(50)
        assert c.tiles > 0 and np.array_equal(c.get_spins(), d.get_spins())
