"""What the paired steps hold besides single steps' arrays, and that it goes
back where they do not run."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
P, W = 1, 0
LAT = (24, 12, 40)
VELOCITIES = [(0.02, -0.01, 0.03), (0.0, 0.04, 0.0), (-0.03, 0.0, 0.01), (0.01, 0.01, -0.02), (0.0, -0.02, 0.02)]


def _fields(plates, gap=3):
    """Plates of 2 x 2 x 3 cells in a row along i, `gap` cells of fluid between
    them (with one, the sites there reach two of them)."""
    phase, vel = np.ones(LAT, dtype=np.uint8), np.zeros(LAT + (3,))
    for b in range(plates):
        at = (slice(1 + (2 + gap) * b, 3 + (2 + gap) * b), slice(3, 5), slice(4, 7))
        phase[at] = 0
        vel[at] = VELOCITIES[b]
    return phase, vel


def _engine(plates, layout="rows", precision="fp64", gap=3):
    from jyulb import _native
    e = _native.Engine(LAT, 1, 0.05, (1e-5, 0.0, 0.0), (P, P, W, W, P, P), precision=precision, layout=layout)
    phase, vel = _fields(plates, gap)
    e.upload_phase(phase)
    e.upload_den_vel(np.ones(LAT), vel)
    e.finalize()
    return e


def _bytes(e):
    return e.info()["device_bytes"]


@pytest.mark.parametrize("layout", ["rows", "sparse"])
@pytest.mark.parametrize("plates,gap,pairs", [(4, 3, True), (5, 2, False), (2, 1, False)],
                         ids=["four_velocities", "five_velocities", "two_at_one_site"])
def test_walls_that_keep_single_steps_hold_nothing(plates, gap, pairs, layout, monkeypatch):
    monkeypatch.setenv("LB_PAIR", "0")
    single = _engine(plates, layout, gap=gap)
    single.evolve(6)
    monkeypatch.setenv("LB_PAIR", "1")
    e = _engine(plates, layout, gap=gap)
    e.evolve(6)
    assert e.paired_steps() == pairs
    assert (_bytes(e) > _bytes(single)) == pairs
    np.testing.assert_array_equal(e.download_post_f(), single.download_post_f())


def test_walls_that_come_to_differ_give_it_back(monkeypatch):
    """Velocities that change between calls: one, then two at one site, then
    one again."""
    out = []
    for pair in ("0", "1"):
        monkeypatch.setenv("LB_PAIR", pair)
        e = _engine(2, gap=1)
        solid = _fields(2, gap=1)[0] == 0
        for scale, pairs in ((0.0, True), (1.0, False), (0.0, True)):
            vel = np.zeros(LAT + (3,))
            vel[solid] = (0.01, 0.02, 0.0)
            vel[4:][solid[4:]] *= 1.0 + scale  # the second plate's
            e.upload_den_vel(np.ones(LAT), vel)
            e.refresh_walls()
            e.evolve(5)
            if pair == "1":
                assert e.paired_steps() == pairs
            out.append(e.download_post_f())
    for a, b in zip(out[:3], out[3:]):
        np.testing.assert_array_equal(b, a)


def test_capture_gives_it_back(monkeypatch):
    import torch
    monkeypatch.setenv("LB_PAIR", "0")
    single = _engine(1)
    monkeypatch.setenv("LB_PAIR", "1")
    e = _engine(1)
    st = torch.cuda.Stream()
    e.set_stream(st.cuda_stream)
    with torch.cuda.stream(st):
        e.evolve(4)
        torch.cuda.synchronize()
        assert _bytes(e) > _bytes(single)
        g = torch.cuda.CUDAGraph()
        g.capture_begin()
        e.evolve(2)
        g.capture_end()
        g.replay()
        e.evolve(2)
        torch.cuda.synchronize()
    single.evolve(8)
    assert _bytes(e) == _bytes(single)
    np.testing.assert_array_equal(e.download_post_f(), single.download_post_f())


def _single(calls, monkeypatch):
    monkeypatch.setenv("LB_PAIR", "0")
    e = _engine(1)
    for n in calls:
        e.evolve(n)
    monkeypatch.setenv("LB_PAIR", "1")
    return e


def test_another_handle_gets_it_back(monkeypatch):
    """An allocation that the device cannot hold takes what the other handles'
    pairs hold before it fails; they go on with single steps."""
    from jyulb import _native
    single = _single((4, 5), monkeypatch)
    e = _engine(1)
    e.evolve(4)
    assert _bytes(e) > _bytes(single)
    with pytest.raises(RuntimeError, match="hipMalloc"):  # 320 GB of populations
        _native.Engine((1290, 1290, 1280), 1, 0.05, (0.0, 0.0, 0.0), (P,) * 6, layout="rows")
    assert _bytes(e) == _bytes(single) and not e.paired_steps()
    e.evolve(5)
    np.testing.assert_array_equal(e.download_post_f(), single.download_post_f())


def test_own_allocation_gets_it_back(monkeypatch):
    """The adjoint's checkpoints on walls at rest."""
    monkeypatch.setenv("LB_PAIR", "1")
    e = _engine(0)
    e.evolve(4)
    held = _bytes(e)
    with pytest.raises(RuntimeError, match="hipMalloc"):
        e.adj_forward(1 << 20, 1, 1, 0)  # terabytes
    assert _bytes(e) < held and not e.paired_steps()
    f = e.download_post_f()
    e.evolve(3)
    assert not np.array_equal(e.download_post_f(), f)


def test_handles_in_other_threads_keep_theirs_while_they_use_it(monkeypatch):
    """Handles stepping in two threads while a third one's allocations fail."""
    import threading
    from jyulb import _native
    calls = [6] * 40
    single = _single(calls, monkeypatch)
    engines = [_engine(1) for _ in range(2)]

    def steps(e):
        for n in calls:
            e.evolve(n)
            e.synchronize()

    def fail():
        for _ in range(10):
            try:
                _native.Engine((1290, 1290, 1280), 1, 0.05, (0.0, 0.0, 0.0), (P,) * 6, layout="rows")
            except RuntimeError:
                pass

    threads = [threading.Thread(target=steps, args=(e,)) for e in engines] + [threading.Thread(target=fail)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for e in engines:
        np.testing.assert_array_equal(e.download_post_f(), single.download_post_f())


def test_pairs_leave_a_quarter_of_the_device_free(monkeypatch):
    """Where less would be left, steps are single, whether the memory goes
    before or after the set-up; LB_PAIR=1 does not ask."""
    import torch
    monkeypatch.delenv("LB_PAIR", raising=False)
    free = _engine(0)
    free.evolve(4)
    assert free.paired_steps()
    late = _engine(0)
    total = torch.cuda.mem_get_info()[1]
    fill = torch.empty(int(0.8 * total), dtype=torch.uint8, device="cuda")
    try:
        early = _engine(0)
        early.evolve(4)
        late.evolve(4)
        assert not early.paired_steps() and not late.paired_steps()
        assert _bytes(early) == _bytes(late) < _bytes(free)
        monkeypatch.setenv("LB_PAIR", "1")
        forced = _engine(0)
        forced.evolve(4)
        assert forced.paired_steps()
    finally:
        del fill
        torch.cuda.empty_cache()
    for e in (early, late, forced):
        np.testing.assert_array_equal(e.download_post_f(), free.download_post_f())


def test_checkpoint_interval_does_not_depend_on_pairs(monkeypatch):
    """interval='auto' budgets the free memory: here of a device that holds 60
    population arrays, of which the pairs' is one."""
    import torch
    from types import SimpleNamespace
    from jyulb import adjoint
    monkeypatch.setenv("LB_PAIR", "1")
    e = _engine(0)
    single = _bytes(e)
    array = 19 * 8 * LAT[0] * LAT[1] * 64
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda: (60 * array - (_bytes(e) - single), 1 << 38))
    solver = SimpleNamespace(engine=e)
    before = [adjoint.checkpoint_interval(solver, n) for n in range(50, 600, 50)]
    assert e.pair_bytes() == 0
    e.evolve(6)
    assert e.pair_bytes() == _bytes(e) - single > 0
    assert [adjoint.checkpoint_interval(solver, n) for n in range(50, 600, 50)] == before
