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
