"""The three forms of the fitting trajectory (all states kept; checkpoints with a segment's predicted spins;
checkpoints alone), with segments that are replayed from a recording and segments that run as launches: the
same magnetisation and gradients bit for bit, whatever form came before in the context."""
import numpy as np
import pytest

from vampire_amd import _lib as L
from vampire_amd import system as S
from vampire_amd.fit import Trajectory

pytestmark = pytest.mark.gpu

HZ = (0.0, 0.0, 1.0)


def _inputs(n, seed):
    rng = np.random.default_rng(seed)
    g = rng.standard_normal((3, n)) * 0.4
    g[2] += 1.0
    return g / np.sqrt((g * g).sum(axis=0)), 0.05 * rng.standard_normal((3, n))


def _same(a, b):
    return all(np.array_equal(np.asarray(x), np.asarray(y)) for x, y in zip(a, b))


@pytest.mark.parametrize("precision,real", [("fp64", 8), ("fp32", 4)])
@pytest.mark.parametrize("crystal,size,topology", [("bcc", 5, "auto"), ("fcc", 4, "ell"), ("sc", 7, "csr")])
def test_forms_give_the_same_gradients(gpu, crystal, size, topology, precision, real):
    s = S.ferromagnet(crystal, size)
    spins, h = _inputs(s.n, 3)
    w = np.linspace(-1.0, 1.5, 25)

    def run(t):
        return (t.forward(S.J_CO, S.KU_CO, 0.1, h), *t.backward(w))

    out = {}
    for K in (37, 100, 250, 400):                    # replays and a remainder; two and one; launches alone
        state = 3 * real * s.n
        for form, limit in ((0, None), (1, 2 * K * state), (2, 0)):
            if form == 1 and K >= 250:
                continue                             # a segment as long as the trajectory: the whole fits too
            t = Trajectory(s, spins, nsteps=250, record_every=10, checkpoint_every=K, H=HZ, precision=precision,
                           topology=topology, resident_bytes=limit)
            assert t.form == -1
            out[K, form] = run(t)
            assert t.form == form
            assert _same(run(t), out[K, form]) and _same(t.backward(w), out[K, form][1:])
            t.close()
    ref = out[100, 0]
    for got in out.values():
        assert _same(got, ref)
    t = Trajectory(s, spins, nsteps=250, record_every=10, checkpoint_every=100, H=HZ, precision=precision, topology=topology)
    for limit, form in ((8 << 30, 0), (0, 2), (200 * state, 1), (8 << 30, 0), (0, 2), (8 << 30, 0)):
        L.check(t.ctx.lib.vmx_fit_set_resident(t.ctx.h, limit))
        assert _same(run(t), ref) and t.form == form
    t.close()


def test_more_records_in_a_segment_than_a_grid_takes(gpu):
    """70,000 recorded states summed in launches of at most 32,768."""
    s = S.ferromagnet("sc", 2)
    spins, _ = _inputs(s.n, 5)
    out = []
    for limit in (None, 0):
        t = Trajectory(s, spins, nsteps=70_000, checkpoint_every=70_000, H=HZ, resident_bytes=limit)
        out.append(t.forward(S.J_CO, S.KU_CO, 0.1))
        assert t.form == (0 if limit is None else 2)
        t.close()
    assert np.array_equal(out[0], out[1]) and np.unique(out[0]).size > 1000
