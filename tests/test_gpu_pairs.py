"""Paired steps (two fused steps per pass over the population array, k_pair) against
the reference's fixtures and against single steps: every boundary kind, tiles
whose edges fall anywhere, and every count of steps."""
import glob
import json
import os

import numpy as np
import pytest

import scenarios

pytestmark = pytest.mark.gpu
GOLD = sorted(glob.glob(os.path.join(os.path.dirname(__file__), "golden", "*.npz")))


def _solver_cls():
    from jyulb.isothermal import Solver
    return Solver


@pytest.mark.parametrize("layout", ["rows", "soa", "sparse"])
@pytest.mark.parametrize("tile", ["", "5,3,2", "3,4,1"], ids=["auto", "5x3x2", "3x4x1"])
@pytest.mark.parametrize("path", GOLD, ids=[os.path.basename(p)[:-4] for p in GOLD])
def test_pairs_bit_exact(path, tile, layout, monkeypatch):
    """FP64 paired steps reproduce the reference bit for bit: periodic, wall,
    symmetric and Zou-He faces, moving walls, in tiles of the engine's choice
    and in small ones with remainders on every axis."""
    monkeypatch.setenv("LB_PAIR", "1")
    if tile:
        monkeypatch.setenv("LB_PAIR_TILE", tile)
    z = np.load(path)
    sc = json.loads(str(z["scenario"]))
    Solver = _solver_cls()
    out = scenarios.run_scenario(lambda *a: Solver(*a, layout=layout), sc, record_f=True)
    fluid = z["sites"].astype(np.int64) + 1
    for k in z.files:
        if k in ("scenario", "nfluid", "sites") or k.startswith("tsteps"):
            continue
        a, b = z[k], out[k]
        if k.startswith("f_"):
            a, b = a[:, fluid[0], fluid[1], fluid[2]], b[:, fluid[0], fluid[1], fluid[2]]
        np.testing.assert_array_equal(b, a, err_msg=f"{sc['name']} {k} tile {tile}")


def _run(lat, bc, precision, rlx, steps, walls, seed, layout="rows", solid=0.04):
    rng = np.random.default_rng(seed)
    s = _solver_cls()(np.array(lat, dtype=np.int32), rlx, 0.05, np.array([1e-5, 2e-5, -1e-5]),
                      np.array(bc, dtype=np.int32), precision=precision, layout=layout)
    phase = (rng.random(lat) > solid).astype(np.uint8)
    s.get_phase()[...] = phase
    s.get_den()[...] = 1.0 + 0.01 * rng.standard_normal(lat)
    s.get_vel()[...] = 0.01 * rng.standard_normal(lat + (3,))
    solid = phase == 0
    s.get_vel()[solid] = 0.0
    if walls == 1:  # every solid site, one velocity
        s.get_vel()[solid] = (0.02, -0.01, 0.03)
    elif walls == 2:  # two velocities; sites between two such walls keep single steps
        s.get_vel()[solid] = np.where(rng.random((solid.sum(), 1)) > 0.5, (0.02, -0.01, 0.03), (0.0, 0.01, 0.0))
    s.finalize_init()
    for n in steps:
        s.evolve(n)
    return s.post_collision_f(), np.array(s.den), np.array(s.vel)


P, W, D, V, S = 1, 0, 2, 3, 4


@pytest.mark.parametrize("precision", ["fp64", "fp32", "fp16", "fp32_storage"])
@pytest.mark.parametrize("lat,bc,tile,walls", [
    ((9, 7, 63), (P, P, P, P, P, P), "16,3,4", 0),      # remainders on every axis, periodic rims
    ((1, 5, 65), (P, P, W, W, P, P), "65,5,1", 1),      # one plane, which is its own neighbour
    ((2, 1, 64), (W, W, P, P, W, W), "", 2),            # one row; a tile from wall to wall along k
    ((33, 18, 34), (P, P, W, S, S, W), "33,9,8", 0),    # mirrors at one end of each axis
    ((12, 40, 130), (W, W, S, S, P, P), "", 1),
    ((21, 11, 16), (V, D, W, W, S, W), "16,5,20", 2),   # Zou-He planes at both ends of the sweep
])
def test_pairs_equal_single_steps(lat, bc, tile, walls, precision, monkeypatch):
    """Pairs change no bit in any precision, whatever the tile and the count
    of steps (a call with an odd count ends in a single step, and the next
    one starts there)."""
    out = []
    for pair in ("0", "1"):
        monkeypatch.setenv("LB_PAIR", pair)
        if tile:
            monkeypatch.setenv("LB_PAIR_TILE", tile)
        print(f"pairs {pair}: {lat} {bc} tile {tile or 'auto'} walls {walls} {precision}", flush=True)
        out.append(_run(lat, bc, precision, 1, (2, 7, 1, 4), walls, 3))
    for a, b, what in zip(*out, ("f", "den", "vel")):
        np.testing.assert_array_equal(b, a, err_msg=what)


@pytest.mark.parametrize("precision", ["fp64", "fp32", "fp16", "fp32_storage"])
@pytest.mark.parametrize("lat,bc,tile,walls,solid", [
    ((9, 7, 63), (P, P, P, P, P, P), "16,3,4", 0, 0.3),
    ((2, 1, 64), (P, P, P, P, W, W), "", 1, 0.1),       # one row, its own neighbour; the planes too
    ((33, 18, 34), (P, P, W, S, S, W), "11,5,8", 0, 0.2),
    ((7, 13, 150), (W, W, S, S, P, P), "", 2, 0.1),
    ((21, 11, 16), (V, D, W, W, S, W), "16,5,20", 2, 0.1),
    ((5, 3, 400), (P, P, P, P, P, P), "200,1,5", 0, 0.97),  # rows and planes without a fluid site
])
def test_sparse_pairs_equal_single_steps(lat, bc, tile, walls, solid, precision, monkeypatch):
    """The same in the sparse layout, from a few solid cells to nearly all,
    against the rows layout's single steps."""
    out = []
    for pair in ("0", "1"):
        monkeypatch.setenv("LB_PAIR", pair)
        if tile:
            monkeypatch.setenv("LB_PAIR_TILE", tile)
        print(f"sparse pairs {pair}: {lat} {bc} tile {tile or 'auto'} walls {walls} {precision}", flush=True)
        out.append(_run(lat, bc, precision, 1, (2, 7, 1, 4), walls, 3, "sparse" if pair == "1" else "rows", solid))
    for a, b, what in zip(*out, ("f", "den", "vel")):
        np.testing.assert_array_equal(b, a, err_msg=what)
