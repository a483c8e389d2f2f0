"""Host fields read and written by the kernels themselves (pinned memory)
against the staged copies that other memory takes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
P, W, D, V, S = 1, 0, 2, 3, 4


def _run(lat, bc, precision, seed):
    from jyulb.isothermal import Solver
    from jyulb.defs import TRT
    rng = np.random.default_rng(seed)
    s = Solver(np.array(lat, dtype=np.int32), TRT, 0.05, np.array([1e-5, 0.0, 2e-5]), np.array(bc, dtype=np.int32),
               precision=precision)
    s.get_phase()[...] = rng.random(lat) > 0.1
    solid = s.get_phase() == 0
    s.get_den()[...] = 1.0 + 0.01 * rng.standard_normal(lat)
    s.get_vel()[...] = 0.01 * rng.standard_normal(lat + (3,))
    s.get_vel()[solid] = 0.0
    s.finalize_init()
    out = []
    for steps in (1, 2, 5):
        s.evolve(steps)
        out.append((np.array(s.den), np.array(s.vel), s.post_collision_f()))
        # between calls: halos and solid sites hold what the user puts there,
        # walls start to move, Ladd's term reads an edited density, a force acts
        s.den[0, :, :] += 0.5
        s.vel[:, -1, :, 1] = 0.25
        s.get_den()[solid] = 3.0 + steps
        s.get_vel()[solid] += 0.01
        s.get_den()[~solid] *= 1.001
        s.get_acc()[0, 0, :, 2] = 1e-4 * steps
    return out


@pytest.mark.parametrize("precision", ["fp64", "fp32", "fp16", "fp32_storage"])
@pytest.mark.parametrize("lat,bc", [((5, 4, 7), (P, P, P, P, P, P)), ((4, 6, 65), (W, W, S, W, P, P)),
                                    ((7, 3, 128), (V, D, W, W, S, S)), ((3, 1, 64), (W, W, P, P, W, S))])
def test_pinned_fields_equal_staged_ones(lat, bc, precision, monkeypatch):
    from jyulb import _native
    pinned = _run(lat, bc, precision, 5)
    monkeypatch.setattr(_native, "host_array", lambda shape, dtype, fill: np.full(shape, fill, dtype=dtype))
    staged = _run(lat, bc, precision, 5)
    for n, (a, b) in enumerate(zip(pinned, staged)):
        for x, y, what in zip(a, b, ("den", "vel", "f")):
            np.testing.assert_array_equal(x, y, err_msg=f"{what} after call {n}")


@pytest.mark.parametrize("lat", [(97, 85, 23), (97, 85, 24), (128, 64, 3), (683, 12, 2)])
def test_short_rows_equal_staged_ones(lat, monkeypatch):
    """Both sides of the lines between staged copies and fields reached in place:
    the length of the rows and their number."""
    test_pinned_fields_equal_staged_ones(lat, (P, P, W, W, S, S), "fp32", monkeypatch)
