"""When single or paired steps are chosen: what the timing compares, and what
settles the choice again."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
P, W = 1, 0
LAT = (24, 20, 40)
TIMED = "paired steps "  # "[jyulb] single steps .. ms, paired steps .. ms per step"


class Flow:
    """A channel with two plates of which the user sets the velocities."""

    def __init__(self, monkeypatch, precision="fp64", layout="rows", **env):
        from jyulb import _native
        monkeypatch.setenv("LB_AUTOTUNE_VERBOSE", "1")
        for k in ("LB_PAIR", "LB_AUTOTUNE", "LB_FP16_CHECK"):
            monkeypatch.delenv(k, raising=False)
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        self.e = _native.Engine(LAT, 1, 0.05, (1e-5, 0.0, 0.0), (P, P, W, W, P, P), precision=precision, layout=layout)
        self.phase = np.ones(LAT, dtype=np.uint8)
        self.phase[4:6, 5:7, 8:11] = 0
        self.phase[7:9, 5:7, 8:11] = 0
        self.e.upload_phase(self.phase)

    def walls(self, first, second):
        vel = np.zeros(LAT + (3,))
        vel[4:6, 5:7, 8:11] = first
        vel[7:9, 5:7, 8:11] = second
        self.e.upload_den_vel(np.ones(LAT), vel)
        return self

    def log(self, capfd, steps):
        capfd.readouterr()
        self.e.evolve(steps)
        out = capfd.readouterr().err
        print(out)
        return out


STILL, SAME, OTHER = (0.0, 0.0, 0.0), (0.02, 0.01, 0.0), (0.0, 0.02, 0.0)


def test_walls_that_do_not_qualify_wait_for_the_timing(monkeypatch, capfd):
    """Two velocities at one site: there is nothing to compare. Once they
    agree, the next long call times both."""
    s = Flow(monkeypatch).walls(SAME, OTHER)
    s.e.finalize()
    assert TIMED not in s.log(capfd, 60)
    assert not s.e.paired_steps() and s.e.pair_bytes() == 0
    s.walls(SAME, SAME).e.refresh_walls()
    assert TIMED not in s.log(capfd, 20)  # too short
    assert TIMED in s.log(capfd, 60)
    assert s.e.paired_steps() == (s.e.pair_bytes() > 0)


@pytest.mark.parametrize("precision,kept", [("fp64", True), ("fp32", False)])
def test_walls_that_start_to_move_settle_it_again(precision, kept, monkeypatch, capfd):
    """Pairs go on where they are never slower (FP64); else both are timed."""
    s = Flow(monkeypatch, precision).walls(STILL, STILL)
    s.e.finalize()
    assert TIMED not in s.log(capfd, 60) and s.e.paired_steps()
    s.walls(SAME, SAME).e.refresh_walls()
    assert s.e.paired_steps() == kept
    assert (TIMED in s.log(capfd, 60)) != kept
    assert s.e.paired_steps() or not kept
    s.walls(STILL, STILL).e.refresh_walls()
    assert s.e.paired_steps()
    assert TIMED not in s.log(capfd, 60)


def test_finalized_again_settles_it_again(monkeypatch, capfd):
    s = Flow(monkeypatch, "fp16").walls(SAME, SAME)
    for _ in range(3):
        s.e.finalize()
        assert not s.e.paired_steps()
        assert TIMED in s.log(capfd, 60)
        assert TIMED not in s.log(capfd, 60)


def test_no_pairs_where_every_step_is_checked(monkeypatch):
    s = Flow(monkeypatch, "fp16", LB_PAIR="1", LB_FP16_CHECK="1").walls(STILL, STILL)
    s.e.finalize()
    s.e.evolve(6)
    assert not s.e.paired_steps() and s.e.pair_bytes() == 0


def test_no_pairs_where_their_array_finds_no_room_in_the_timing(monkeypatch, capfd):
    import torch
    s = Flow(monkeypatch, "fp16").walls(STILL, STILL)
    s.e.finalize()
    fill = torch.empty(int(0.8 * torch.cuda.mem_get_info()[1]), dtype=torch.uint8, device="cuda")
    try:
        assert TIMED in s.log(capfd, 60)
    finally:
        del fill
        torch.cuda.empty_cache()
    assert not s.e.paired_steps() and s.e.pair_bytes() == 0


@pytest.mark.parametrize("since", [0, 30, 50, 63])
@pytest.mark.parametrize("velocity", [STILL, SAME], ids=["still", "moving"])
def test_fp16_checks_stay_where_they_were(since, velocity, monkeypatch, capfd):
    """The timing waits for the next check of the FP16 values, and changes no
    bit: the same steps with LB_PAIR=0."""
    out = []
    for env in ({"LB_PAIR": "0"}, {}):
        s = Flow(monkeypatch, "fp16", **env).walls(velocity, velocity)
        s.e.finalize()
        for _ in range(since):
            s.e.evolve(1)
        log = s.log(capfd, 60) + s.log(capfd, 70)
        assert (TIMED in log) == (not env)
        out.append((s.e.download_post_f(), *s.e.download_den_vel(), s.e.info()["fp16_scale"]))
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
