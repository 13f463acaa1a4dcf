"""The workloads this framework is measured on: what a spin-dynamics program has it do, through the
public entry points (vampire_amd.context.Context, vampire_amd.fit.Trajectory), over the sizes that
the benchmark, the tests and such programs use.

``listed()`` gives the fixed cases, ``draw(rng)`` more of the same ranges.  ``prepare`` builds the
context a program keeps (system uploaded, spins set, statistics registered, colouring done), ``run``
is one pass: a stretch of the simulation and what the program takes from it, the spins among it.
``exact`` forms the same numbers in 64 bits with plain torch.

The results of an FP32 context are returned as float32: its spins and fields are floats, and the
doubles that the interface hands over hold nothing beyond them.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from vampire_amd import system as S
from vampire_amd.context import FP32, FP64, Context
from vampire_amd.fit import Trajectory

H_APPLIED = (0.0, 0.05, 0.4)      # T; a field off the easy axis, as a field-cooled or FMR run has it
FIT_H = (0.0, 0.0, 1.0)           # T; the fitting workload's field
ANGLES = (40.0, 30.0)             # degrees; constraint direction of the constrained sweeps


def listed():
    return [
        # The reference's own CPU-sized run: SC 20^3 at 300 K in double precision, many steps replayed
        # from one graph, spins read at the end.  8000 atoms: every launch is short.
        dict(name="heun_sc20_fp64_graph", kind="heun", crystal="sc", nx=20, ny=20, nz=20, precision=FP64, T=300.0,
             steps=1000, mode="graph", stats=0),
        # The smallest calls: a program that drives the device as VAMPIRE's gpu:: interface does, setting
        # the conditions before each single step and updating its statistics every tenth.
        dict(name="steps_sc9_fp64", kind="heun", crystal="sc", nx=9, ny=9, nz=9, precision=FP64, T=300.0, steps=50,
             mode="each", stats=10),
        # The benchmark workload: FCC 100^3 (4M atoms) in single precision, a magnetisation and an energy
        # every hundred steps, spins read at the end.
        dict(name="heun_fcc100_fp32", kind="heun", crystal="fcc", nx=100, ny=100, nz=100, precision=FP32, T=600.0,
             steps=1000, mode="eager", stats=100),
        # The same crystal in double precision at an odd, middling size (1.0M atoms).
        dict(name="heun_fcc63_fp64", kind="heun", crystal="fcc", nx=63, ny=63, nz=63, precision=FP64, T=600.0,
             steps=200, mode="eager", stats=50),
        # The midpoint integrator on an odd BCC block (208k atoms).
        dict(name="midpoint_bcc47_fp32", kind="heun", crystal="bcc", nx=47, ny=47, nz=47, precision=FP32, T=300.0,
             steps=200, mode="midpoint", stats=50),
        # A diluted two-material film with interfacial DMI (3x3 exchange tensors, irregular rows) under a
        # laser pulse: the temperature is set before every step.
        dict(name="film_dmi_pulse_fp32", kind="film", nx=256, ny=256, nz=8, precision=FP32, steps=200, stats=50),
        # An M(T) curve in one context: replicas of ragged sizes, each at its own temperature, LLG steps
        # replayed from a graph.
        dict(name="replicas_llg_fp32", kind="replicas", count=64, lmin=8, lmax=48, precision=FP32, steps=200),
        # The same curve by checkerboard Metropolis: one call of many sweeps.
        dict(name="replicas_mc_fp32", kind="mc", count=64, lmin=8, lmax=48, precision=FP32, sweeps=50, each=0),
        # A single odd lattice swept as VAMPIRE's gpu::mc_step does: one sweep a call, statistics after each.
        dict(name="mc_sc33_fp64_each", kind="mc", count=1, lmin=33, lmax=33, precision=FP64, sweeps=20, each=1),
        # Constrained Monte Carlo on a batch (anisotropy against temperature).
        dict(name="replicas_cmc_fp32", kind="cmc", count=24, lmin=8, lmax=48, precision=FP32, sweeps=20),
        # Fitting J, Ku, damping and site fields to a trajectory: forward and adjoint, BCC 32^3.
        dict(name="fit_bcc32_fp32", kind="fit", L=32, precision=FP32, steps=2000, record=10, checkpoint=100),
        # A film with its macrocell dipole field refreshed on the device every ten steps (768 cells).
        dict(name="dipole_film_fp64", kind="dipole", nx=64, ny=64, nz=10, cell=4, precision=FP64, steps=100, rate=10),
    ]


# ---- drawn cases ----------------------------------------------------------------------------------
def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _precision(rng):
    return FP32 if rng.random() < 0.6 else FP64


def draw(rng):
    kind = rng.choice(["heun", "heun", "heun", "midpoint", "film", "replicas", "mc", "mc", "cmc", "fit", "dipole"])
    prec = _precision(rng)
    if kind in ("heun", "midpoint"):
        crystal = rng.choice(["sc", "bcc", "fcc"])
        basis = {"sc": 1, "bcc": 2, "fcc": 4}[crystal]
        mode = "midpoint" if kind == "midpoint" else rng.choice(["eager", "graph", "each"])
        atoms = _log_int(rng, 500, 3_000_000 if prec == FP32 else 1_500_000)
        side = max(3, (atoms / basis) ** (1.0 / 3.0))
        nx, ny = (max(3, int(round(side * rng.uniform(0.7, 1.4)))) for _ in range(2))
        nz = max(3, int(round(atoms / basis / (nx * ny))))
        if mode == "graph":
            steps = 100 * rng.randint(1, 5)
        elif mode == "each":
            steps = rng.randint(50, 120)
        else:
            steps = rng.randint(100, 500)
        return dict(kind="heun", crystal=crystal, nx=nx, ny=ny, nz=nz, precision=prec,
                    T=round(rng.uniform(10.0, 900.0), 1), steps=steps, mode=mode,
                    stats=0 if mode == "graph" else rng.choice([10, 25, 50]))
    if kind == "film":
        return dict(kind="film", nx=_log_int(rng, 24, 256), ny=_log_int(rng, 24, 256), nz=rng.randint(3, 8),
                    precision=prec, steps=rng.randint(50, 200), stats=rng.choice([10, 50]))
    if kind == "replicas":
        lmin = rng.randint(6, 16)
        return dict(kind="replicas", count=rng.randint(4, 48), lmin=lmin, lmax=lmin + rng.randint(2, 30), precision=prec,
                    steps=50 * rng.randint(1, 4))
    if kind == "mc":
        if rng.random() < 0.5:
            L = _log_int(rng, 7, 90)
            return dict(kind="mc", count=1, lmin=L, lmax=L, precision=prec, sweeps=rng.randint(5, 30),
                        each=1 if rng.random() < 0.5 else 0)
        lmin = rng.randint(6, 16)
        return dict(kind="mc", count=rng.randint(4, 48), lmin=lmin, lmax=lmin + rng.randint(2, 30), precision=prec,
                    sweeps=rng.randint(5, 50), each=0)
    if kind == "cmc":
        lmin = rng.randint(6, 16)
        return dict(kind="cmc", count=rng.randint(1, 24), lmin=lmin, lmax=lmin + rng.randint(2, 30), precision=FP32,
                    sweeps=rng.randint(1, 20))
    if kind == "fit":
        record = rng.choice([5, 10, 20])
        return dict(kind="fit", L=_log_int(rng, 5, 36), precision=prec, steps=record * rng.randint(300 // record, 1200 // record),
                    record=record, checkpoint=rng.choice([50, 75, 100]))
    cell = rng.randint(2, 5)
    return dict(kind="dipole", nx=cell * rng.randint(4, 16), ny=cell * rng.randint(4, 16), nz=rng.randint(2, 12), cell=cell,
                precision=prec, steps=rng.randint(40, 120), rate=rng.choice([5, 10, 20]))


# ---- systems --------------------------------------------------------------------------------------
# The lattices do not depend on the seed; spins, noise, temperatures of a run do.
@functools.lru_cache(maxsize=3)
def _block(crystal, nx, ny, nz, pbc_z=True):
    alpha = 0.05 if crystal == "fcc" else 0.1
    return S.ferromagnet(crystal, nx, alpha=alpha, Ly=ny, Lz=nz, pbc=(True, True, pbc_z))


@functools.lru_cache(maxsize=2)
def _film(nx, ny, nz):
    return S.config_c4(nx, ny, nz)


@functools.lru_cache(maxsize=2)
def _replicas(count, lmin, lmax):
    systems, temps = S.config_c2(count, L_min=lmin, L_max=lmax)
    return (S.concat_systems(systems) if count > 1 else systems[0]), tuple(temps)


def _tilted(n, seed, spread=0.4):
    """Spins about +z with a thermal spread: a magnet below its Curie temperature."""
    g = np.random.default_rng(seed).standard_normal((3, n))
    g *= spread
    g[2] += 1.0
    g /= np.sqrt((g * g).sum(axis=0))
    return g


def _system(case):
    kind = case["kind"]
    if kind == "heun":
        return _block(case["crystal"], case["nx"], case["ny"], case["nz"])
    if kind == "film":
        return _film(case["nx"], case["ny"], case["nz"])
    if kind == "dipole":
        return _block("sc", case["nx"], case["ny"], case["nz"], False)
    if kind == "fit":
        return _block("bcc", case["L"], case["L"], case["L"])
    return _replicas(case["count"], case["lmin"], case["lmax"])[0]


def _temperatures(case, seed):
    """Replica temperatures of a case: the batch's spread over [0, 1.5 Tc], or one near 300 K."""
    system, temps = _replicas(case["count"], case["lmin"], case["lmax"])
    if case["count"] == 1:
        return [300.0]
    shift = (seed * 0.61803398875) % 1.0
    top = 1.5 * S.TC_SC_CO
    return [(t + shift * top) % top for t in temps]


def _pulse(case):
    """Electron temperature of a laser pulse, 300 K to 1200 K, sampled at every step."""
    k = np.arange(case["steps"])
    return [300.0 + 900.0 * math.exp(-((i - case["steps"] / 2) / (case["steps"] / 5)) ** 2) for i in k]


def _cells(case):
    """Macrocells of cell^3 lattice sites: cell of each atom, cell volumes and the dipole tensor
    (3 r r - 1) / r^3 between cell centres (A^-3), as the tensor method's set-up leaves it."""
    system = _system(case)
    a = 3.54
    edge = case["cell"] * a
    dims = [-(-case[k] // case["cell"]) for k in ("nx", "ny", "nz")]
    ijk = np.floor(system.coords / edge + 1e-9).astype(np.int64)
    atom_cell = (ijk[:, 0] * dims[1] + ijk[:, 1]) * dims[2] + ijk[:, 2]
    nc = dims[0] * dims[1] * dims[2]
    count = np.bincount(atom_cell, minlength=nc)
    centre = np.stack([np.bincount(atom_cell, system.coords[:, k], nc) / count for k in range(3)], axis=1)
    r = centre[None, :, :] - centre[:, None, :]
    d2 = (r * r).sum(axis=2)
    np.fill_diagonal(d2, 1.0)
    inv3 = d2 ** -1.5
    tensor = np.empty((6, nc, nc))
    for k, (p, q) in enumerate(((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))):
        tensor[k] = (3.0 * r[..., p] * r[..., q] / d2 - (1.0 if p == q else 0.0)) * inv3
        np.fill_diagonal(tensor[k], 0.0)
    return dict(num_cells=nc, local_cell=np.arange(nc, dtype=np.int32), atom_cell=atom_cell.astype(np.int32),
                volume=count * a ** 3, tensor=tensor, update_rate=case["rate"])


# ---- what a program holds before the pass -----------------------------------------------------------
def prepare(case, seed):
    system = _system(case)
    kind = case["kind"]
    state = dict(case=case, system=system, fp32=case["precision"] == FP32)
    if kind == "fit":
        state.update(_fit_inputs(case, seed))
        state["traj"] = Trajectory(system, state["spins"], nsteps=case["steps"], record_every=case["record"],
                                   checkpoint_every=case["checkpoint"], precision=case["precision"], H=FIT_H)
        return state
    ctx = Context(system, precision=case["precision"], seed=seed, device=0)
    state["ctx"] = ctx
    if kind in ("heun", "film"):
        if case["stats"]:
            # the system's magnetisation, or each material's (the last mask id collects non-magnetic atoms)
            state["mag"] = ctx.add_magnetization(system.type, len(system.materials) + 1)
            state["energy"] = ctx.add_energy(np.zeros(system.n, np.int32), 2)
        ctx.set_conditions(case.get("T", 300.0), H_APPLIED)
        ctx.set_spins(_tilted(system.n, seed))
    elif kind == "dipole":
        ctx.set_conditions(300.0, H_APPLIED)
        ctx.set_spins(_tilted(system.n, seed))
        ctx.set_dipole(**_cells(case))
    else:
        for r, T in enumerate(_temperatures(case, seed)):
            ctx.set_conditions(T, replica=r)
        ctx.set_spins(_tilted(system.n, seed))
        if kind == "cmc":
            ctx.cmc_set_constraint(*ANGLES)
            ctx.mc_set_sigma(0.3)
            ctx.mc_num_colours()
        elif kind == "mc":
            if case["each"]:
                state["mag"] = ctx.add_magnetization(np.zeros(system.n, np.int32), 2)
            ctx.mc_set_sigma(0.5)
            ctx.mc_num_colours()
    ctx.synchronize()
    return state


def _fit_inputs(case, seed):
    system = _system(case)
    rng = np.random.default_rng(seed)
    theta = np.radians(30.0 + 8.0 * rng.standard_normal(system.n))
    phi = 0.3 * rng.standard_normal(system.n)
    spins = np.stack([np.sin(theta) * np.cos(phi), np.sin(theta) * np.sin(phi), np.cos(theta)])
    t = np.arange(1, case["steps"] // case["record"] + 1) * case["record"] / 2000.0
    return dict(spins=spins, h=0.01 * rng.standard_normal((3, system.n)), target=0.85 + 0.05 * t + 0.01 * rng.random(),
                J=S.J_CO * rng.uniform(0.9, 1.1), Ku=S.KU_CO * rng.uniform(0.8, 1.2), alpha=rng.uniform(0.08, 0.14))


# ---- one pass -----------------------------------------------------------------------------------------
def _held(state, *arrays):
    """What the context's precision holds of its results."""
    return [torch.from_numpy(a).float() if state["fp32"] else a for a in arrays]


def _statistics(state):
    ctx = state["ctx"]
    m, m_sum, _ = ctx.magnetization(state["mag"])
    out = [m, m_sum]
    if "energy" in state:
        e, e_sum, _ = ctx.energy(state["energy"])
        out += [e, e_sum]
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "fit":
        traj = state["traj"]
        mz = traj.forward(state["J"], state["Ku"], state["alpha"], state["h"])
        dJ, dKu, da, dh = traj.backward(2.0 * (mz - state["target"]) / mz.size)
        # the loss's sensitivity to a relative change of each parameter, and to each site field
        return _held(state, mz, np.array([dJ * state["J"], dKu * state["Ku"], da * state["alpha"]]), dh)
    ctx = state["ctx"]
    if kind in ("heun", "film"):
        steps, stats = case["steps"], case["stats"]
        if stats:
            ctx.stats_reset()
        if kind == "film" or case["mode"] == "each":
            temps = _pulse(case) if kind == "film" else None
            for k in range(steps):
                ctx.set_conditions(temps[k] if temps else case["T"], H_APPLIED)
                ctx.llg_heun(1)
                if stats and (k + 1) % stats == 0:
                    ctx.stats_update()
        elif case["mode"] == "graph":
            ctx.llg_heun_graph(100, steps // 100)
        else:
            advance = ctx.llg_midpoint if case["mode"] == "midpoint" else ctx.llg_heun
            done = 0
            while done < steps:
                k = min(stats, steps - done)
                advance(k)
                ctx.stats_update()
                done += k
        return _held(state, ctx.get_spins(), *(_statistics(state) if stats else []))
    if kind == "replicas":
        ctx.llg_heun_graph(50, case["steps"] // 50)
        return _held(state, ctx.get_spins())
    if kind == "dipole":
        ctx.llg_heun(case["steps"])
        return _held(state, ctx.get_spins(), *ctx.dipole_field())
    if kind == "cmc":
        ctx.cmc_sweep(case["sweeps"])
        return _held(state, ctx.get_spins()) + [ctx.cmc_counts().astype(np.int64)]
    if case["each"]:
        ctx.stats_reset()
        for _ in range(case["sweeps"]):
            ctx.mc_sweep(1)
            ctx.stats_update()
    else:
        ctx.mc_sweep(case["sweeps"])
    sigma, moves, rejects = ctx.mc_state()
    out = _held(state, ctx.get_spins(), sigma, *(_statistics(state) if case["each"] else []))
    return out + [moves.astype(np.int64), rejects.astype(np.int64)]


# ---- what a pass cannot do without ----------------------------------------------------------------------
def work(case):
    """Bytes: every stage of a step or sweep reads the spins it starts from and writes the ones it makes
    once (materials, stencils and tables are small), and the pass hands the spins over as doubles.
    Flops: exchange, random numbers and the update, per atom and stage."""
    system = _system(case)
    n, p = system.n, (4 if case["precision"] == FP32 else 8)
    z = system.nnz / n
    k = {1: 1, 3: 3, 9: 9}[system.exchange.shape[1]]
    exchange = 2 * z * (3 if k <= 3 else 9)
    kind = case["kind"]
    if kind == "fit":
        # forward: S, P, S_next; adjoint: states, adjoint vectors and site-field gradient in and out
        return dict(bytes=float(n * p * case["steps"] * (12 + 24)), flops=float(n * case["steps"] * (4 * exchange + 400)))
    if kind in ("mc", "cmc"):
        return dict(bytes=float(n * (case["sweeps"] * 6 * p + 24)), flops=float(n * case["sweeps"] * (2 * exchange + 150)))
    bytes_, flops = n * (case["steps"] * 15 * p + 24.0), n * case["steps"] * (2 * exchange + 300.0)
    if kind == "dipole":
        nc = np.prod([-(-case[d] // case["cell"]) for d in ("nx", "ny", "nz")])
        refreshes = case["steps"] // case["rate"]
        bytes_ += refreshes * (6.0 * nc * nc * 8 + n * (3 * p + 6 * 8.0))
        flops += refreshes * 18.0 * nc * nc
    return dict(bytes=float(bytes_), flops=float(flops))


# ---- the same in 64 bits, plain torch ---------------------------------------------------------------------
def _philox(c0, step, stream, key):
    """Philox-4x32-10 (Salmon et al., SC'11) of the counters (c0, step, 0, stream), words in int64."""
    mask = 0xFFFFFFFF
    k0, k1 = key & mask, (key >> 32) & mask
    c = [c0, torch.full_like(c0, step & mask), torch.full_like(c0, (step >> 32) & mask), torch.full_like(c0, stream)]
    for r in range(10):
        p0, p1 = c[0] * 0xD2511F53, c[2] * 0xCD9E8D57
        hi0, hi1 = (p0 >> 32) & mask, (p1 >> 32) & mask
        c = [hi1 ^ c[1] ^ ((k0 + r * 0x9E3779B9) & mask), p1 & mask, hi0 ^ c[3] ^ ((k1 + r * 0xBB67AE85) & mask), p0 & mask]
    return c


def _normals(words):
    u = [(w.double() + 0.5) * 2.0 ** -32 for w in words]
    r1, r2 = torch.sqrt(-2.0 * torch.log(u[0])), torch.sqrt(-2.0 * torch.log(u[2]))
    t1, t2 = 2.0 * math.pi * u[1], 2.0 * math.pi * u[3]
    return torch.stack([r1 * torch.cos(t1), r1 * torch.sin(t1), r2 * torch.cos(t2)])


class _Exact:
    """One system in 64 bits: fields, steps, sweeps and statistics."""

    def __init__(self, system, seed):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=self.dev)  # noqa: E731
        self.s, self.n = system, system.n
        deg = (system.nbr_end - system.nbr_start + 1).astype(np.int64)
        self.z = int(deg.max())
        slot = np.arange(self.z)
        pos = np.where(slot < deg[:, None], system.nbr_start[:, None] + slot, 0)
        self.valid = t(slot < deg[:, None])
        self.nbr = torch.where(self.valid, t(system.nbr[pos].astype(np.int64)), torch.zeros(1, dtype=torch.int64, device=self.dev))
        J = t(system.exchange)
        self.k = J.shape[1]
        if self.k == 1 and bool((J == J[0]).all()):
            self.J = J[0, 0] * self.valid.double()
        else:
            ids = t(system.nbr_iid[pos].astype(np.int64))
            self.J = J[ids] * self.valid[..., None].double()       # [n, z, k]
            self.J = self.J[..., 0] if self.k == 1 else self.J
        off = system.replica_offset if system.replica_offset is not None else np.array([0, system.n])
        rep = np.repeat(np.arange(len(off) - 1), np.diff(off))
        self.nrep, self.rep = len(off) - 1, t(rep)
        self.local = t(np.arange(system.n) - off[rep])
        self.key = t(rep) + int(seed) if self.nrep > 1 else int(seed)
        self.type = t(system.type.astype(np.int64))
        mat = lambda f: torch.tensor([m[f] for m in system.materials], dtype=torch.float64, device=self.dev)  # noqa: E731
        self.a, self.b = mat("one_oneplusalpha_sq")[self.type], mat("alpha_oneplusalpha_sq")[self.type]
        self.alpha, self.ku = mat("alpha")[self.type], mat("ku2")[self.type] * (system.anisotropy_flags & 1)
        self.width, self.mu = mat("H_th_sigma")[self.type], mat("mu_s_SI")[self.type]
        self.axis = torch.tensor(system.materials[0]["ku_vector"], dtype=torch.float64, device=self.dev)[:, None]
        self.moment = t(system.moment)
        self.extra = None

    def conditions(self, temps, H):
        self.T = torch.tensor(temps, dtype=torch.float64, device=self.dev)[self.rep] if len(temps) > 1 else temps[0]
        self.H = torch.tensor(H, dtype=torch.float64, device=self.dev)[:, None]
        self.sigma = self.width * (torch.sqrt(self.T) if torch.is_tensor(self.T) else math.sqrt(self.T))

    def exchange(self, sp):
        out = torch.zeros_like(sp)
        for k in range(self.z):
            g = sp[:, self.nbr[:, k]]
            if self.k == 9:
                j = self.J[:, k]
                out += torch.stack([j[:, 0] * g[0] + j[:, 1] * g[1] + j[:, 2] * g[2],
                                    j[:, 3] * g[0] + j[:, 4] * g[1] + j[:, 5] * g[2],
                                    j[:, 6] * g[0] + j[:, 7] * g[1] + j[:, 8] * g[2]])
            else:
                out += self.J[:, k] * g
        return out

    def field(self, sp):
        return self.exchange(sp) + 2.0 * self.ku * (sp * self.axis).sum(0) * self.axis

    def external(self, step):
        ext = _normals(_philox(self.local, step, 0, self.key)) * self.sigma + self.H
        return ext if self.extra is None else ext + self.extra

    def rhs(self, sp, h):
        g = torch.cross(sp, h, dim=0)
        return self.a * g + self.b * torch.cross(sp, g, dim=0)

    def heun(self, sp, step):
        ext, dt = self.external(step), self.s.dt
        d = self.rhs(sp, self.field(sp) + ext)
        p = sp + dt * d
        p = p / p.norm(dim=0)
        d2 = self.rhs(p, self.field(p) + ext)
        out = sp + self.s.half_dt * (d + d2)
        return out / out.norm(dim=0)

    def midpoint(self, sp, step):
        ext, beta = self.external(step), -0.5 * self.s.dt * self.a

        def rotate(m, h):
            f = h + self.alpha * torch.cross(m, h, dim=0)
            ff, fs = (f * f).sum(0), (f * sp).sum(0)
            return (sp * (1 - beta ** 2 * ff) + 2 * (beta * torch.cross(f, sp, dim=0) + beta ** 2 * fs * f)) / (1 + beta ** 2 * ff)

        m = 0.5 * (sp + rotate(sp, self.field(sp) + ext))
        return rotate(m, self.field(m) + ext)

    def energies(self, sp, H):
        w = self.moment
        ex = -(self.exchange(sp) * sp).sum(0)
        an = -self.ku * (sp * self.axis).sum(0) ** 2
        ap = -(torch.tensor(H, dtype=torch.float64, device=self.dev)[:, None] * sp).sum(0)
        ex, an, ap = 0.5 * float((ex * w).sum()), float((an * w).sum()), float((ap * w).sum())
        return np.array([ex + an + ap, ex, an, ap, 0.0])

    def magnetisation(self, sp, mask, bins):
        out = np.zeros(4 * bins)
        for b in range(bins - 1):
            w = self.moment * (mask == b)
            m = (sp * w).sum(1)
            out[4 * b:4 * b + 3] = (m / m.norm()).cpu().numpy()
            out[4 * b + 3] = float(m.norm() / w.sum())
        return out

    def colours(self):
        """The greedy colouring in atom order."""
        nbr, deg = self.nbr.cpu().tolist(), self.valid.sum(1).cpu().tolist()
        c = [-1] * self.n
        for i in range(self.n):
            used = {c[j] for j in nbr[i][:deg[i]]}
            k = 0
            while k in used:
                k += 1
            c[i] = k
        c = torch.tensor(c, device=self.dev)
        return [torch.nonzero(c == k)[:, 0] for k in range(int(c.max()) + 1)]

    def sweep(self, sp, sweep, colours, width):
        """A checkerboard Metropolis sweep of one replica; returns the number of rejected moves."""
        rejected = 0
        scale = self.mu * 1.07828231e23 * 9.27400915e-24 / (self.T * 1.3806503e-23)
        for atoms in colours:
            old = sp[:, atoms]
            new = old + width * _normals(_philox(self.local[atoms], sweep, 1, self.key))
            new = new / new.norm(dim=0)
            h = torch.zeros_like(old)
            for k in range(self.z):
                h += self.J[atoms, k] * sp[:, self.nbr[atoms, k]]
            e = [-(h * v).sum(0) - self.ku[atoms] * (v * self.axis).sum(0) ** 2 - (self.H * v).sum(0) for v in (old, new)]
            x = (e[1] - e[0]) * scale[atoms]
            u = _philox(self.local[atoms], sweep, 2, self.key)[0].double() * 2.0 ** -32
            take = (x < 0) | (torch.exp(-x) >= u)
            sp[:, atoms] = torch.where(take, new, old)
            rejected += int((~take).sum())
        return rejected


def exact(case, seed):
    kind = case["kind"]
    if kind == "cmc" or (kind == "mc" and (case["precision"] == FP32 or case["count"] > 1)):
        # A Markov chain that accepts its moves in single precision is another chain than the 64-bit one;
        # and a batch's colouring is a sequential walk over millions of atoms.
        return None
    system = _system(case)
    if kind == "fit":
        return _exact_fit(case, seed, system)
    x = _Exact(system, seed)
    sp = torch.as_tensor(_tilted(system.n, seed), device=x.dev)
    host = lambda a: a.cpu().numpy()  # noqa: E731
    if kind == "mc":
        return _exact_mc(case, x, sp)
    if kind == "replicas":
        x.conditions(_temperatures(case, seed), (0.0, 0.0, 0.0))
        for k in range(case["steps"]):
            sp = x.heun(sp, k)
        return [host(sp)]
    x.conditions([case.get("T", 300.0)], H_APPLIED)
    if kind == "dipole":
        cells = _cells(case)
        b, hd = _dipole(x, sp, cells)
        for k in range(case["steps"]):
            x.extra = b
            sp = x.heun(sp, k)
            if (k + 1) % case["rate"] == 0:
                b, hd = _dipole(x, sp, cells)
        return [host(sp), host(b), host(hd)]
    temps = _pulse(case) if kind == "film" else None
    advance = x.midpoint if kind == "heun" and case["mode"] == "midpoint" else x.heun
    bins = len(system.materials) + 1
    m_sum, e_sum, m, e = np.zeros(4 * bins), np.zeros((5, 2)), None, None
    updates_at_end = kind == "heun" and case["mode"] in ("eager", "midpoint")
    for k in range(case["steps"]):
        if temps:
            x.conditions([temps[k]], H_APPLIED)
        sp = advance(sp, k)
        if case["stats"] and ((k + 1) % case["stats"] == 0 or (updates_at_end and k + 1 == case["steps"])):
            m = x.magnetisation(sp, x.type, bins)
            # the last mask id collects what is not magnetic: no atoms, no energy
            e = np.stack([x.energies(sp, H_APPLIED), np.zeros(5)], axis=1)
            m_sum, e_sum = m_sum + m, e_sum + e
    return [host(sp)] + ([m, m_sum, e, e_sum] if case["stats"] else [])


def _exact_mc(case, x, sp):
    x.conditions([300.0], (0.0, 0.0, 0.0))
    colours, width = x.colours(), 0.5
    moves = rejects = 0
    m, m_sum = None, np.zeros(8)
    for w in range(case["sweeps"]):
        r = x.sweep(sp, w, colours, width)
        moves, rejects = moves + x.n, rejects + r
        width = width * (0.5 / (r / x.n)) if r else 60.0
        width = 60.0 if width > 60.0 or width < 1e-5 else width
        m = x.magnetisation(sp, torch.zeros_like(x.type), 2)
        m_sum = m_sum + m
    out = [sp.cpu().numpy(), np.array([width])] + ([m, m_sum] if case["each"] else [])
    return out + [np.array([moves]), np.array([rejects])]


def _dipole(x, sp, cells):
    """Cell moments, cell fields and their values at the atoms: B and mu0 Hd (T)."""
    t = lambda a, d=torch.float64: torch.as_tensor(np.asarray(a), dtype=d, device=x.dev)  # noqa: E731
    cell, nc = t(cells["atom_cell"], torch.int64), cells["num_cells"]
    mag = torch.zeros((3, nc), dtype=torch.float64, device=x.dev).index_add_(1, cell, sp * x.mu) / S.MU_B
    T = t(cells["tensor"])
    rows = ((0, 1, 2), (1, 3, 4), (2, 4, 5))
    b = torch.stack([sum(T[rows[r][q]] @ mag[q] for q in range(3)) for r in range(3)])
    hd = b - 0.5 * 8.0 * math.pi / (3.0 * t(cells["volume"])) * mag
    return 0.927400915 * b[:, cell], 0.927400915 * hd[:, cell]


def _exact_fit(case, seed, system):
    """Trajectory and gradient by automatic differentiation, segments recomputed in the backward pass."""
    from torch.utils.checkpoint import checkpoint
    inp = _fit_inputs(case, seed)
    x = _Exact(system, 0)
    mu = system.materials[0]["mu_s_SI"]
    gamma, dt = system.materials[0]["gamma_rel"], system.dt
    leaf = lambda v: torch.tensor(v, dtype=torch.float64, device=x.dev, requires_grad=True)  # noqa: E731
    J, Ku, alpha, h = leaf(inp["J"] / mu), leaf(inp["Ku"] / mu), leaf(inp["alpha"]), leaf(inp["h"])
    H = torch.tensor(FIT_H, dtype=torch.float64, device=x.dev)[:, None]
    nbr = x.nbr.reshape(-1)

    def rhs(sp, J, Ku, alpha, h):
        f = J * sp[:, nbr].view(3, x.n, x.z).sum(2) + 2.0 * Ku * (sp * x.axis).sum(0) * x.axis + H + h
        a = -gamma / (1.0 + alpha * alpha)
        g = torch.cross(sp, f, dim=0)
        return a * g + alpha * a * torch.cross(sp, g, dim=0)

    def segment(sp, J, Ku, alpha, h):
        for _ in range(case["record"]):
            d = rhs(sp, J, Ku, alpha, h)
            p = sp + dt * d
            p = p / p.norm(dim=0)
            sp = sp + system.half_dt * (d + rhs(p, J, Ku, alpha, h))
            sp = sp / sp.norm(dim=0)
        return sp

    sp = torch.as_tensor(inp["spins"], device=x.dev)
    mz = []
    for _ in range(case["steps"] // case["record"]):
        sp = checkpoint(segment, sp, J, Ku, alpha, h, use_reentrant=False)
        mz.append(sp[2].mean())
    mz = torch.stack(mz)
    target = torch.as_tensor(inp["target"], device=x.dev)
    ((mz - target) ** 2).mean().backward()
    par = torch.stack([J.grad * J, Ku.grad * Ku, alpha.grad * alpha]).detach()
    return [mz.detach().cpu().numpy(), par.cpu().numpy(), h.grad.cpu().numpy()]
