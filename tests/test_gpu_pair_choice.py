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
