"""Paired steps in lattices that are known to take them: every case says
whether it steps in pairs, and is refused if it does otherwise. Moving walls
with Zou-He faces, mirror faces and a force field in every precision and
collision, and the palette of wall velocities up to its size and beyond it."""
import json
import os

import numpy as np
import pytest

import scenarios

pytestmark = pytest.mark.gpu
P, W, D, V, S = 1, 0, 2, 3, 4
PRECISIONS = ["fp64", "fp32", "fp16", "fp32_storage"]
# wall velocities of the palette; the fifth does not fit
VELOCITIES = [(0.02, -0.01, 0.03), (0.0, 0.04, 0.0), (-0.03, 0.0, 0.01), (0.01, 0.01, -0.02), (0.0, -0.02, 0.02)]


def _blocks(n, lat, rng):
    """n plates of 2 x 2 x 3 cells in a row along i, three cells of fluid
    between them and two to every face: no site reaches two of them, nor one
    through a mirror."""
    solid, vel = np.zeros(lat, dtype=bool), np.zeros(lat + (3,))
    for b in range(n):
        at = (slice(3 + 5 * b, 5 + 5 * b), slice(3, 5), slice(4, 7))
        solid[at] = True
        vel[at] = VELOCITIES[b]
    return solid, vel


def _still(lat, rng):
    return rng.random(lat) < 0.05, np.zeros(lat + (3,))


def _split(n, lat, rng):
    """Two plates side by side: the sites between them see both velocities."""
    solid, vel = _blocks(1, lat, rng)
    solid[6:8, 3:5, 4:7] = True
    vel[6:8, 3:5, 4:7] = VELOCITIES[1]
    return solid, vel


# name: lattice, faces, tile, plates, force field, whether steps are paired
KINDS = {
    "zouhe_x": ((21, 11, 16), (V, D, W, W, S, W), "16,5,20", 0, False, True),
    "zouhe_x_ends": ((9, 10, 66), (D, V, P, P, W, W), "24,4,3", 0, True, True),
    "zouhe_y": ((7, 12, 40), (P, P, V, D, W, W), "20,5,4", 0, False, True),
    "zouhe_z": ((10, 9, 33), (W, W, P, P, D, D), "11,4,5", 0, False, True),
    "plate": ((14, 9, 40), (P, P, P, P, W, W), "14,4,3", 1, False, True),
    "plate_force": ((14, 9, 40), (P, P, P, P, W, W), "14,4,3", 1, True, True),
    "plate_mirrors": ((9, 10, 70), (W, W, S, S, S, S), "24,5,4", 1, False, True),
    "plates_zouhe_mirrors_force": ((14, 9, 35), (V, D, W, S, S, W), "12,5,4", 2, True, True),
    "plates_zouhe_y": ((14, 9, 34), (P, P, D, V, P, P), "", 2, False, True),
    "plates_3": ((19, 8, 20), (W, W, S, W, P, P), "10,3,5", 3, False, True),
    "plates_4": ((24, 8, 13), (P, P, P, P, P, P), "", 4, True, True),
    "plates_5": ((29, 8, 13), (P, P, P, P, P, P), "", 5, False, False),
    "split": ((14, 9, 40), (P, P, P, P, W, W), "", -1, False, False),
    "mirror_x": ((9, 7, 20), (S, W, W, W, P, P), "", 0, False, False),
}


def _run(kind, precision, rlx, layout, expect=None, calls=(2, 7, 1, 4)):
    from jyulb.isothermal import Solver
    lat, bc, tile, plates, force, pairs = KINDS[kind]
    rng = np.random.default_rng(7)
    s = Solver(np.array(lat, dtype=np.int32), rlx, 0.05, np.array([1e-5, 2e-5, -1e-5]), np.array(bc, dtype=np.int32),
               precision=precision, layout=layout)
    solid, vel = (_still(lat, rng) if plates == 0 else _split(1, lat, rng) if plates < 0 else _blocks(plates, lat, rng))
    s.get_phase()[...] = ~solid
    s.get_den()[...] = 1.0 + 0.01 * rng.standard_normal(lat)
    s.get_vel()[...] = 0.01 * rng.standard_normal(lat + (3,))
    s.get_vel()[solid] = vel[solid]
    if force:
        s.get_acc()[...] = 1e-4 * rng.standard_normal(lat + (3,))
    s.finalize_init()
    if expect is not None:
        assert s.engine.paired_steps() == expect
    held = s.engine.info()["device_bytes"]
    for n in calls:
        s.evolve(n)
    if expect is not None:  # they did run: their second array is there
        assert s.engine.paired_steps() == expect
        assert (s.engine.info()["device_bytes"] > held) == expect
    return s.post_collision_f(), np.array(s.den), np.array(s.vel)


def _compare(kind, precision, rlx, layout, monkeypatch):
    lat, bc, tile, plates, force, pairs = KINDS[kind]
    print(f"{kind} {precision} collision {rlx} {layout}", flush=True)
    monkeypatch.setenv("LB_PAIR", "0")
    single = _run(kind, precision, rlx, "rows", expect=False)
    monkeypatch.setenv("LB_PAIR", "1")
    if tile:
        monkeypatch.setenv("LB_PAIR_TILE", tile)
    paired = _run(kind, precision, rlx, layout, expect=pairs)
    for a, b, what in zip(single, paired, ("f", "den", "vel")):
        np.testing.assert_array_equal(b, a, err_msg=f"{kind} {what}")


@pytest.mark.parametrize("layout", ["rows", "sparse"])
@pytest.mark.parametrize("precision", PRECISIONS)
@pytest.mark.parametrize("kind", list(KINDS))
def test_pairs_run_and_equal_single_steps(kind, precision, layout, monkeypatch):
    _compare(kind, precision, 1, layout, monkeypatch)


@pytest.mark.parametrize("layout", ["soa", "sparse"])
@pytest.mark.parametrize("precision", PRECISIONS)
@pytest.mark.parametrize("rlx", [0, 2], ids=["bgk", "reg"])
@pytest.mark.parametrize("kind", ["zouhe_x", "plate", "plates_zouhe_mirrors_force"])
def test_pairs_of_the_other_collisions(kind, rlx, precision, layout, monkeypatch):
    _compare(kind, precision, rlx, layout, monkeypatch)


# Fixtures that step in pairs by themselves, with the single steps' launches:
# they need LB_PAIR=0 to reach the launch tuner and the tile orders.
@pytest.mark.parametrize("env", [{"LB_AUTOTUNE": "1", "LB_AUTOTUNE_MIN_CELLS": "0"}, {"LB_XCD_REMAP_CELLS": "0"}],
                         ids=["tuned", "xcd_order"])
@pytest.mark.parametrize("name", ["c1_poiseuille", "bgk_zouhe_x"])
def test_single_steps_launches_on_lattices_that_pair(name, env, monkeypatch):
    from jyulb.isothermal import Solver
    z = np.load(os.path.join(os.path.dirname(__file__), "golden", name + ".npz"))
    sc = json.loads(str(z["scenario"]))
    monkeypatch.setenv("LB_PAIR", "0")
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    out = scenarios.run_scenario(lambda *a: Solver(*a, layout="rows"), sc, record_f=True)
    fluid = z["sites"].astype(np.int64) + 1
    for k in z.files:
        if k in ("scenario", "nfluid", "sites") or k.startswith("tsteps"):
            continue
        a, b = z[k], out[k]
        if k.startswith("f_"):
            a, b = a[:, fluid[0], fluid[1], fluid[2]], b[:, fluid[0], fluid[1], fluid[2]]
        np.testing.assert_array_equal(b, a, err_msg=f"{name} {k}")


@pytest.mark.parametrize("lat,precision,lid,pairs", [
    ((24, 20, 40), "fp64", True, True),
    ((64, 64, 64), "fp32", True, False), ((66, 64, 64), "fp32", True, True),
    ((64, 64, 256), "fp32_storage", True, False), ((65, 64, 256), "fp32_storage", True, True),
    ((24, 20, 40), "fp16", True, False), ((24, 20, 40), "fp16", False, True),
    ((24, 20, 40), "fp32", False, True), ((24, 20, 40), "fp32_storage", False, True),
    ((256, 128, 128), "fp16", False, True), ((257, 128, 128), "fp16", False, False),
])
def test_untimed_choice(lat, precision, lid, pairs, monkeypatch):
    """LB_AUTOTUNE=0 times nothing: pairs where they are never slower, single
    steps elsewhere, from the first call on."""
    from jyulb import _native
    monkeypatch.delenv("LB_PAIR", raising=False)
    monkeypatch.setenv("LB_AUTOTUNE", "0")
    e = _native.Engine(lat, 1, 0.05, (1e-6, 0.0, 0.0), (P, P, W, W, W, W), precision=precision, layout="rows")
    phase, vel = np.ones(lat, dtype=np.uint8), np.zeros(lat + (3,))
    if lid:
        phase[:, :, -1] = 0
        vel[:, :, -1, 0] = 0.05
    e.upload_phase(phase)
    e.upload_den_vel(np.ones(lat), vel)
    e.finalize()
    held = e.info()["device_bytes"]
    e.evolve(30)
    assert e.paired_steps() == pairs
    assert (e.info()["device_bytes"] > held) == pairs


@pytest.mark.parametrize("lat,precision,layout,pairs", [
    ((1024, 1, 1), "fp64", "rows", True), ((4096, 1, 1), "fp64", "rows", False), ((4096, 2, 4), "fp64", "rows", True),
    ((8192, 2, 4), "fp32_storage", "rows", False), ((8192, 3, 4), "fp32_storage", "rows", True),
    ((4096, 1, 64), "fp32", "soa", False), ((4096, 1, 200), "fp32", "soa", True), ((1, 4096, 1), "fp32", "rows", True),
    ((900, 800, 1), "fp64", "sparse", False), ((1, 800, 900), "fp64", "sparse", False),
    ((420, 4, 420), "fp64", "sparse", True), ((4000, 12, 14), "fp64", "sparse", False),
    ((2800, 16, 16), "fp64", "sparse", True),
])
def test_thin_lattices(lat, precision, layout, pairs, monkeypatch):
    """Lattices of which the planes are too thin for the pairs' sweep step
    singly, and the same bits either way."""
    from jyulb import _native
    rng = np.random.default_rng(2)
    phase = (rng.random(lat) > (0.15 if layout == "sparse" else 0.01)).astype(np.uint8)
    out = []
    for pair in (None, "1", "0"):
        monkeypatch.delenv("LB_PAIR", raising=False)
        if pair:
            monkeypatch.setenv("LB_PAIR", pair)
        print(f"{lat} {precision} {layout} LB_PAIR={pair}", flush=True)
        e = _native.Engine(lat, 1, 0.05, (1e-6, 2e-6, 0.0), (P,) * 6, precision=precision, layout=layout)
        e.upload_phase(phase)
        e.upload_den_vel(1.0 + 0.01 * np.random.default_rng(3).standard_normal(lat), np.zeros(lat + (3,)))
        e.finalize()
        e.evolve(7)
        assert e.paired_steps() == (pairs if pair is None else pair == "1")
        out.append((e.download_post_f(), *e.download_den_vel()))
    for a, b, c in zip(*out):
        np.testing.assert_array_equal(a, c)
        np.testing.assert_array_equal(b, c)
