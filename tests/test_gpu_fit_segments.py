"""The fitting trajectory at the edges of its segments (50 steps are recorded and replayed, the rest runs
as launches), with and without a kept trajectory, against automatic differentiation of the same step in
64-bit torch: relative 1e-9 of each output's norm (a few hundred steps of rounding at 1e-16)."""
import numpy as np
import pytest
import torch

from vampire_amd import system as S
from vampire_amd.fit import Trajectory

pytestmark = pytest.mark.gpu

HZ = (0.0, 0.1, 1.0)


def _inputs(n, seed):
    rng = np.random.default_rng(seed)
    g = rng.standard_normal((3, n)) * 0.4
    g[2] += 1.0
    return g / np.sqrt((g * g).sum(axis=0)), 0.05 * rng.standard_normal((3, n))


def _autograd(s, spins, h, J, Ku, alpha, nsteps, record, weights):
    mu = s.materials[0]["mu_s_SI"]
    leaf = lambda v: torch.tensor(v, dtype=torch.float64, requires_grad=True)  # noqa: E731
    J, Ku, alpha, h = leaf(J / mu), leaf(Ku / mu), leaf(alpha), leaf(h)
    z = int((s.nbr_end[0] - s.nbr_start[0]) + 1)
    nbr = torch.as_tensor(s.nbr.astype(np.int64))
    axis = torch.tensor(s.materials[0]["ku_vector"], dtype=torch.float64)[:, None]
    H = torch.tensor(HZ, dtype=torch.float64)[:, None]

    def rhs(sp):
        f = J * sp[:, nbr].view(3, s.n, z).sum(2) + 2.0 * Ku * (sp * axis).sum(0) * axis + H + h
        a = -1.0 / (1.0 + alpha * alpha)
        g = torch.cross(sp, f, dim=0)
        return a * g + alpha * a * torch.cross(sp, g, dim=0)

    sp, mz = torch.as_tensor(spins), []
    for q in range(nsteps):
        d = rhs(sp)
        p = sp + s.dt * d
        p = p / p.norm(dim=0)
        sp = sp + s.half_dt * (d + rhs(p))
        sp = sp / sp.norm(dim=0)
        if (q + 1) % record == 0:
            mz.append(sp[2].mean())
    mz = torch.stack(mz)
    (mz * torch.as_tensor(weights)).sum().backward()
    return mz.detach().numpy(), (J.grad / mu).item(), (Ku.grad / mu).item(), alpha.grad.item(), h.grad.numpy()


def _close(a, b, tol=1e-9):
    a, b = np.asarray(a), np.asarray(b)
    assert np.linalg.norm(a - b) <= tol * np.linalg.norm(b), (np.linalg.norm(a - b), np.linalg.norm(b))


@pytest.mark.parametrize("crystal,L,topology", [("bcc", 3, "auto"), ("sc", 7, "csr"), ("fcc", 4, "ell")])
@pytest.mark.parametrize("nsteps,record", [(1, 1), (49, 7), (50, 50), (51, 17), (99, 3), (100, 20), (153, 9)])
def test_segment_edges_against_autograd(gpu, crystal, L, topology, nsteps, record):
    s = S.ferromagnet(crystal, L)
    spins, h = _inputs(s.n, 3)
    w = np.linspace(-1.0, 1.5, nsteps // record)
    t = Trajectory(s, spins, nsteps=nsteps, record_every=record, checkpoint_every=30, H=HZ, topology=topology)
    for k in range(3):                              # the third call replays what the second recorded
        J, Ku, alpha = S.J_CO * (1 + 0.1 * k), S.KU_CO * (1 - 0.2 * k), 0.1 + 0.02 * k
        hk = h * (1 + k)
        mz = t.forward(J, Ku, alpha, hk)
        dJ, dKu, da, dh = t.backward(w)
        ref = _autograd(s, spins, hk, J, Ku, alpha, nsteps, record, w)
        for got, want in zip((mz, dJ, dKu, da, dh), ref):
            _close(got, want)
    t.close()


def test_checkpoints_when_the_trajectory_does_not_fit(gpu):
    """2800 steps of 65,536 FP64 atoms are 8.8 GB of states: checkpoints and recomputation, at two
    distances, give the same gradient bit for bit; FP32 (4.4 GB, kept) agrees with them to its precision."""
    s = S.config_c3()
    spins, h = _inputs(s.n, 4)
    out = []
    for precision, every in (("fp64", 100), ("fp64", 37), ("fp32", 100)):
        t = Trajectory(s, spins, nsteps=2800, record_every=100, checkpoint_every=every, precision=precision, H=HZ)
        mz = t.forward(S.J_CO, S.KU_CO, 0.1, h)
        out.append((mz, *t.backward(np.linspace(-1.0, 1.0, mz.size))))
        t.close()
    for a, b in zip(out[0], out[1]):
        assert np.array_equal(a, b)
    for a, b in zip(out[2], out[0]):
        _close(a, b, 1e-3)
