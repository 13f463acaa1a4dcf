"""The library's host logic on a HIP runtime that computes nothing (tests/host): what is launched with what,
what is allocated, and what happens when a call fails.  No GPU."""
import pytest

from host import fake


@pytest.fixture(scope="module")
def hip(tmp_path_factory):
    return fake.build(tmp_path_factory.mktemp("fakehip"))


@pytest.mark.parametrize("kernel,argument,L", [("k_tile_step", 6, 6), ("k_fused_predictor", 7, 42)])
def test_conditions_outlive_a_launch_that_failed(hip, kernel, argument, L):
    """Conditions that a launch was to carry to the device table stay with the context when it fails: the
    next step carries them (the same values set again write nothing, so nothing else would)."""
    fake.run(hip, f"""
        s = S.ferromagnet("sc", {L})
        hip.fake_watch(b"{kernel}", {argument})              # CondArg: its first word, the words carried
        with Context(s, precision=FP32, seed=1) as c:
            c.set_spins(S.random_spins(s.n, 2))
            c.llg_heun(s.n // 128 + 1)
            c.set_conditions(300.0)
            hip.fake_fail_launch(b"{kernel}", 1)
            try:
                c.llg_heun(1)
                assert 0, "the launch was to fail"
            except L.VmxError:
                pass
            c.set_conditions(300.0)
            carried = [l.watched[0] for l in launches(log(lambda: c.llg_heun(2)), "{kernel}")]
            assert carried[0] > 0 and carried[1] == 0, carried
    """)


@pytest.mark.parametrize("n", [200_000, 750_001])            # one worker, several
@pytest.mark.parametrize("to_host", [True, False])
@pytest.mark.parametrize("nth", [1, 2, 3])
def test_a_transfer_that_failed_leaves_no_copy_in_flight(hip, n, to_host, nth):
    """Copies still queued would write into the slots (or read from them) while the next transfer uses them."""
    fake.run(hip, f"""
        s = RC.isolated_spins({n})
        with Context(s, precision=FP64, seed=1) as c:
            sp = S.random_spins(s.n, 2)
            c.set_spins(sp)

            def fails():
                hip.fake_fail_copy({nth})
                try:
                    c.get_spins() if {to_host} else c.set_spins(sp)
                    assert 0, "the transfer was to fail"
                except L.VmxError:
                    pass
            lines = log(fails)
            queued = max(k for k, x in enumerate(lines) if x.startswith("copy"))
            assert "wait stream" in lines[queued:], lines[-8:]
            c.set_spins(sp)
            assert c.get_spins().shape == sp.shape
    """)


def test_a_segment_of_many_records_is_summed_within_the_grid_limit(hip):
    """A checkpoint distance of 100,000 steps with every step recorded: 100,000 records in one segment, and a
    grid's second dimension holds 65,535."""
    fake.run(hip, """
        from vampire_amd.fit import Trajectory
        s = S.ferromagnet("sc", 16)
        steps = 100_000                                       # 19.7 GB of states: checkpoints
        t = Trajectory(s, S.random_spins(s.n, 2), nsteps=steps, record_every=1, checkpoint_every=steps)
        got = launches(log(lambda: t.forward(S.J_CO, S.KU_CO, 0.1)), "k_fit_mz")
        assert sum(l.grid[1] for l in got) == steps and max(l.grid[1] for l in got) <= 65535, [l.grid for l in got]
        t.close()
    """)


DIPOLE = """
        def dipole(cells, n):
            return dict(num_cells=cells, local_cell=np.arange(cells), atom_cell=np.arange(n) % cells,
                        volume=np.ones(cells), tensor=np.zeros((6, cells, cells)), update_rate=1)
"""


def test_a_dipole_tensor_needs_its_own_memory_once(hip):
    """Setting the dipole field takes the tensor in the device's layout and a small buffer beside it, not the
    caller's layout whole as well."""
    fake.run(hip, DIPOLE + """
        s = RC.isolated_spins(2001)
        cells = 1501
        tensor = 6 * 8 * cells * cells
        with Context(s, precision=FP64, seed=1) as c:
            hip.fake_capacity(hip.fake_used() + tensor + tensor // 2)
            c.set_dipole(**dipole(cells, s.n))
    """)


def test_a_dipole_field_that_cannot_be_set_leaves_none(hip):
    """The tables of an earlier field are overwritten one by one: when one finds no memory, no step may form a
    field from the mixture."""
    fake.run(hip, DIPOLE + """
        s = RC.isolated_spins(2001)
        with Context(s, precision=FP64, seed=1) as c:
            c.set_conditions(0.0)
            c.set_dipole(**dipole(11, s.n))
            assert launches(log(lambda: c.llg_heun(1)), "k_dip_field")
            hip.fake_capacity(hip.fake_used() + (4 << 20))
            try:
                c.set_dipole(**dipole(501, s.n))
                assert 0, "there was to be no memory"
            except L.VmxError as e:
                assert e.code == L.VMX_ERR_NOMEM
            assert not launches(log(lambda: c.llg_heun(1)), "k_dip")
            try:
                c.dipole_field()
                assert 0, "no field is set"
            except L.VmxError as e:
                assert e.code == L.VMX_ERR_STATE
    """)


@pytest.mark.parametrize("step", ["llg_heun", "llg_midpoint"])
def test_only_rows_that_read_the_staged_exchange_table_stage_it(hip, step):
    """The step kernels of ELL and stencil rows read exchange tables of up to 8 KiB from LDS; those of CSR rows
    read the table itself and stage the material and condition records alone."""
    fake.run(hip, f"""
        s = S.config_c4(16, 16, 5)                    # a film of tensors, more atoms than make tiles at once
        staged = {{}}
        for topology in ("csr", "ell"):
            with Context(s, precision=FP32, seed=1, topology=topology) as c:
                assert c.topology[0] == topology
                c.set_spins(S.random_spins(s.n, 2))
                staged[topology] = sorted(set(l.shared for l in launches(log(lambda: c.{step}(1)), "tor")))
        records, tensors = 4 * 2 * (18 + 12), 4 * 9 * 28     # of the two materials; the film's 28
        assert staged == dict(csr=[records], ell=[records + tensors]), staged
    """)


def test_small_arrays_cross_in_one_copy(hip):
    """A copy on the link costs about 10 us whatever its size: the three components of a small system's spins or
    fields share one, an array going to the device is not waited for, and a tensor of megabytes goes in chunks of
    its own size, not of the system's."""
    fake.run(hip, DIPOLE + """
        s = RC.isolated_spins(1000)
        with Context(s, precision=FP64, seed=1) as c:
            sp = S.random_spins(s.n, 2)
            c.set_spins(sp)
            copies = lambda lines: [x for x in lines if x.startswith("copy")]
            assert copies(log(c.get_spins)) == ["copy 2 24000"]
            assert copies(log(c.fields)) == ["copy 2 24000"] * 2
            lines = log(lambda: c.set_spins(sp))
            assert copies(lines) == ["copy 1 24000"]
            assert sum(x.startswith("wait") for x in lines) == 1, lines     # for the call, not for the slot
            lines = log(lambda: c.set_dipole(**dipole(400, s.n)))
            assert len(copies(lines)) < 60, len(copies(lines))
            assert copies(log(c.dipole_field)) == ["copy 2 19200"]       # the cells' two fields
        s = RC.isolated_spins(43_000)                         # just within a slot
        with Context(s, precision=FP32, seed=1) as c:
            assert copies(log(c.get_spins)) == ["copy 2 1032000"]
    """)


@pytest.mark.parametrize("n", [1, 2731, 21_846, 43_690, 43_691, 50_001, 130_000, 200_000, 750_001])
def test_chunked_transfers_keep_every_value_in_its_place(hip, n):
    """Lengths around a slot (512 KiB to 1 MiB), two and more, and several workers: what the runtime holds after the
    copies is what the caller handed over (the kernels, which would permute, do nothing here)."""
    fake.run(hip, f"""
        s = RC.isolated_spins({n})
        with Context(s, precision=FP64, seed=1) as c:
            for k in range(3):
                sp = np.random.default_rng(k).standard_normal((3, s.n))
                c.set_spins(sp)
                assert np.array_equal(c.get_spins(), sp)      # both go through the staging array
    """)


def test_the_step_takes_the_form_it_reports(hip):
    """tiles is what the next step uses, and two kernels kept means two kernels, eagerly and in a recording."""
    fake.run(hip, """
        s = S.ferromagnet("sc", 13)                           # tiles from the 17th step on
        with Context(s, precision=FP64, seed=1) as c:
            c.set_spins(S.random_spins(s.n, 2))
            whole = lambda call: {l.name.startswith("k_tile_step") for l in launches(log(call))
                                  if re.match("k_(tile_step|fused|mid)", l.name)}
            assert c.tiles == 0 and whole(lambda: c.llg_heun(1)) == {False}
            c.llg_heun(20)
            assert c.tiles > 0
            for run in (lambda: c.llg_heun(1), lambda: c.llg_midpoint(1), lambda: c.llg_heun_graph(2, 1)):
                for on in (False, True):
                    c.set_whole_step(on)
                    assert (c.tiles > 0) == on and whole(run) == {on}
    """)


def test_autotuning_times_the_launch_shape_it_chooses(hip):
    """The workgroup size and remapping shape the two kernels, not the whole-step kernel: every trial is of the
    two, and the trials are not counted towards the tiles."""
    fake.run(hip, """
        s = S.ferromagnet("sc", 13)                           # tiles from the 17th step on
        for made in (False, True):
            with Context(s, precision=FP64, seed=1) as c:
                c.set_spins(S.random_spins(s.n, 2))
                if made:
                    c.llg_heun(20)
                tiles = c.tiles
                assert (tiles > 0) == made
                lines = log(lambda: c.autotune(10))
                assert not launches(lines, "k_tile"), launches(lines, "k_tile")[0].name
                shapes = {(l.grid[0], l.block) for l in launches(lines, "k_fused_corrector")}
                assert len(shapes) == 8 or len({b for _, b in shapes}) == 4, shapes
                assert c.tiles == tiles
                c.llg_heun(16)
                assert (c.tiles > 0) == made
                c.llg_heun(1)
                assert c.tiles > 0
    """)


FIT = """
        from vampire_amd.fit import Trajectory
        s = S.ferromagnet("sc", 16)                           # 4096 atoms, 98,304 bytes a state
        state = 24 * s.n
        sp = S.random_spins(s.n, 2)
        traj = lambda **kw: Trajectory(s, sp, nsteps=1000, record_every=10, checkpoint_every=100, **kw)
        both = lambda t: (t.forward(S.J_CO, S.KU_CO, 0.1), t.backward(np.ones(100)))
        memory = lambda lines: [x for x in lines if x.startswith(("malloc", "free", "capture"))]
"""


def test_the_kept_trajectory_leaves_room_for_the_backward_pass(hip):
    """Where the trajectory alone would fit and the working arrays of the backward pass would not beside it,
    checkpoints are taken: both passes run."""
    fake.run(hip, FIT + """
        for spare in (105, 108, 112, 130):                    # segments and small arrays take 103 states
            t = traj()
            hip.fake_capacity(hip.fake_used() + (2000 + spare) * state)
            both(t)
            print(spare, t.form)
            t.close()
    """)


def test_a_form_that_found_no_memory_is_not_tried_again(hip):
    """Each try would free and allocate the segment, and so record both passes anew."""
    fake.run(hip, FIT + """
        t = traj()
        hip.fake_capacity(hip.fake_used() + 600 * state)
        both(t)
        assert t.form == 1
        both(t)
        assert memory(log(lambda: both(t))) == []
        hip.fake_capacity(288 << 30)
        assert memory(log(lambda: both(t))) == [] and t.form == 1
        L.check(t.ctx.lib.vmx_fit_set_resident(t.ctx.h, 8 << 30))      # asked again
        both(t)
        assert t.form == 0
    """)


def test_checkpoints_bound_the_memory_when_asked_to(hip):
    fake.run(hip, FIT + """
        used = hip.fake_used()
        t = traj(resident_bytes=0)
        base = hip.fake_used() - used
        both(t)
        assert t.form == 2
        states = (hip.fake_used() - used - base) / state      # 10 checkpoints, 101 of a segment, 11 arrays
        assert states < 125, states
        L.check(t.ctx.lib.vmx_fit_set_resident(t.ctx.h, 200 * state))
        both(t)
        assert t.form == 1
        L.check(t.ctx.lib.vmx_fit_set_resident(t.ctx.h, 2000 * state))
        both(t)
        assert t.form == 0
        kept = hip.fake_used()
        L.check(t.ctx.lib.vmx_fit_set_resident(t.ctx.h, 2000 * state - 1))
        both(t)
        assert t.form == 1 and hip.fake_used() <= kept - 2000 * state, (hip.fake_used(), kept)
    """)


def test_an_allocation_done_without_leaves_no_error(hip):
    """Tiles, a kept trajectory and further transfer slots are taken where there is memory for them: a call that
    went on without has nothing to report, and an earlier error's text stays."""
    fake.run(hip, FIT + """
        lib = L.load()
        t = traj()
        hip.fake_capacity(hip.fake_used() + 600 * state)
        t.forward(S.J_CO, S.KU_CO, 0.1)
        assert t.ctx.lib.vmx_last_error() == b""
        hip.fake_capacity(288 << 30)
        t.close()

        def earlier(c):
            assert lib.vmx_mc_set_sigma(c.h, 99, 1.0) == L.VMX_ERR_ARG
            return lib.vmx_last_error()

        with Context(S.ferromagnet("sc", 20), precision=FP64, seed=1) as c:      # no memory for tiles
            c.set_spins(S.random_spins(8000, 2))
            text = earlier(c)
            hip.fake_capacity(hip.fake_used())
            c.llg_heun(100)
            assert text and lib.vmx_last_error() == text, lib.vmx_last_error()
            assert c.tiles == 0
            hip.fake_capacity(288 << 30)
        big = RC.isolated_spins(1_000_001)
        with Context(big, precision=FP64, seed=1) as c:                          # nor for more slots
            text = earlier(c)
            hip.fake_capacity(hip.fake_used())
            c.set_spins(np.zeros((3, big.n)))
            assert lib.vmx_last_error() == text, lib.vmx_last_error()
            hip.fake_capacity(288 << 30)
    """)


@pytest.mark.parametrize("L,folded", [(50, True), (52, False)])
def test_a_constrained_sweeps_first_round_adds_a_bounded_number_of_partials(hip, L, folded):
    """A basis-major crystal has four runs of cells: 7816 and 8788 entries of 64 atoms, around the 8192 that every
    workgroup of the sweep's first round may add; the later rounds' own partials are few either way."""
    fake.run(hip, f"""
        s = S.ferromagnet("fcc", {L})
        with Context(s, precision=FP32, seed=1, block_size=64) as c:
            c.set_conditions(300.0)
            c.set_spins(S.random_spins(s.n, 2))
            c.cmc_set_constraint(10.0, 20.0)
            c.cmc_sweep(1)
            names = [l.name for l in launches(log(lambda: c.cmc_sweep(3)))]
            assert sum("k_cmc_pairs" in x for x in names) == 3 * 8, names
            assert sum("k_moment_finish" in x for x in names) == (0 if {folded} else 3), names
            assert not any("k_moment_add" in x for x in names), names
    """)


def test_a_trajectory_of_one_segment_is_not_copied(hip):
    """50 steps and fewer stay where they were computed: no second copy of the states, in memory or time."""
    fake.run(hip, FIT + """
        for nsteps, copies in ((10, 1), (50, 1), (51, None)):
            t = Trajectory(s, sp, nsteps=nsteps, record_every=1)
            used = hip.fake_used()
            f = log(lambda: t.forward(S.J_CO, S.KU_CO, 0.1))
            b = log(lambda: t.backward(np.ones(nsteps)))
            inside = lambda lines: sum(x.startswith("copy 3") for x in lines)
            assert t.form == 0
            if copies:
                assert inside(f) == inside(b) == copies, (nsteps, inside(f), inside(b))     # the first state
                assert hip.fake_used() - used < (2 * nsteps + 15) * state
            t.close()
    """)


def test_transfers_wait_for_events(hip):
    """hipStreamSynchronize sleeps and may wake milliseconds late; an event is waited for by spinning."""
    fake.run(hip, """
        for n in (100, 60_000, 750_001):                      # one copy, several, several workers
            s = RC.isolated_spins(n)
            with Context(s, precision=FP64, seed=1) as c:
                sp = S.random_spins(n, 2)
                h, e = c.add_magnetization(np.zeros(n, np.int32), 1), c.add_energy(np.zeros(n, np.int32), 2)
                for call in (lambda: c.set_spins(sp), c.get_spins, lambda: c.magnetization(h), lambda: c.energy(e),
                             c.mc_state, c.cmc_counts):
                    lines = log(call)
                    assert any(x.startswith("wait ") for x in lines) and "wait stream" not in lines, lines
    """)
