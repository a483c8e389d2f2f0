"""Evolve steps captured in a HIP graph, replayed between the handle's plain
calls: the graph and the handle keep stepping the same populations."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
P, W = 1, 0


def _engine(lat, bc, precision, layout, solid, lid, stream):
    from jyulb import _native
    e = _native.Engine(lat, 1, 0.05, (1e-5, 0.0, 2e-5), bc, precision=precision, layout=layout)
    rng = np.random.default_rng(3)
    phase = (rng.random(lat) >= solid).astype(np.uint8)
    vel = 0.01 * rng.standard_normal(lat + (3,))
    if lid:
        phase[:, :, -1] = 0
    vel[phase == 0] = (0.05, 0.0, 0.0) if lid else 0.0
    e.upload_phase(phase)
    e.upload_den_vel(np.ones(lat), vel)
    e.finalize()
    e.set_stream(stream.cuda_stream)
    return e


@pytest.mark.parametrize("before", [0, 1, 2, 4], ids=lambda n: f"after_{n}")
@pytest.mark.parametrize("lat,bc,precision,layout,solid,lid", [
    ((24, 20, 64), (P, P, W, W, P, P), "fp64", "rows", 0.0, False),
    ((9, 14, 37), (P, P, W, W, P, P), "fp32", "soa", 0.05, False),
    ((20, 16, 30), (W,) * 6, "fp64", "rows", 0.0, True),         # a lid: paired once they are timed
    ((16, 16, 40), (P,) * 6, "fp64", "sparse", 0.1, False),
], ids=["channel", "soa", "lid", "sparse"])
def test_replays_between_plain_calls(lat, bc, precision, layout, solid, lid, before, monkeypatch):
    """An even number of captured steps, so that every replay starts from the
    parity that the capture saw; plain calls of even and, in pairs, odd counts."""
    import torch
    if not lid:
        monkeypatch.setenv("LB_PAIR", "1")
    st = torch.cuda.Stream()
    e, ref = (_engine(lat, bc, precision, layout, solid, lid, st) for _ in range(2))
    print(f"{lat} {precision} {layout}, captured after {before} steps", flush=True)
    with torch.cuda.stream(st):
        e.evolve(2 * before)
        ref.evolve(2 * before)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        g.capture_begin()
        e.evolve(4)
        g.capture_end()
        for n, plain in enumerate((2, 40, 3, 1, 6)):
            g.replay()
            torch.cuda.synchronize()
            ref.evolve(4)
            e.evolve(plain)
            ref.evolve(plain)
            if plain % 2:  # back to the parity of the capture
                e.evolve(1)
                ref.evolve(1)
            for a, b, what in zip((e.download_post_f(), *e.download_den_vel()),
                                  (ref.download_post_f(), *ref.download_den_vel()), ("f", "den", "vel")):
                np.testing.assert_array_equal(a, b, err_msg=f"{what} after replay {n}")
    assert not e.paired_steps()


@pytest.mark.parametrize("layout,lid", [("rows", False), ("rows", True), ("sparse", False)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_a_captured_call_times_nothing(precision, layout, lid, monkeypatch):
    """A call long enough for the launch tuner and for the timing of pairs,
    captured; then plain ones, which may tune."""
    import torch
    monkeypatch.setenv("LB_AUTOTUNE_MIN_CELLS", "0")
    st = torch.cuda.Stream()
    e, ref = (_engine((20, 16, 30), (W,) * 6, precision, layout, 0.1 if layout == "sparse" else 0.0, lid, st)
              for _ in range(2))
    print(f"{precision} {layout} lid {lid}", flush=True)
    with torch.cuda.stream(st):
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        g.capture_begin()
        e.evolve(80)
        g.capture_end()
        for n, plain in enumerate((80, 2, 100)):
            g.replay()
            torch.cuda.synchronize()
            ref.evolve(80)
            e.evolve(plain)
            ref.evolve(plain)
            np.testing.assert_array_equal(e.download_post_f(), ref.download_post_f(), err_msg=f"after replay {n}")
