"""The rules that shape a list run when nothing sets them: the interval between list-build
opportunities (from a new state's speeds, the time step and the thermostat) and the lanes per
atom (from the number of atoms and of list entries).  NBX_BUILD_EVERY and NBX_LANES stay
unset."""
import math

import numpy as np
import pytest

from nbodysimulator import _lib
from nbodysimulator import generators as gen
from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def defaults(monkeypatch):
    for k in ("NBX_BUILD_EVERY", "NBX_LANES", "NBX_TUNE_CACHE"):
        monkeypatch.delenv(k, raising=False)


def lj_ctx(u, v, L, R=2.5, skin=0.3, thermostat=None):
    ctx = _lib.Context(len(u), _lib.SYS_POTENTIAL, np.ones(len(u)))
    ctx.set_boundary(_lib.BC_CUBIC, [L, 0, 0, 0, 0, 0])
    ctx.add_lennard_jones(1.0, 1.0, R)
    ctx.set_kb(1.0)
    ctx.set_precision(_lib.PREC_MIXED)
    ctx.set_skin(skin)
    if thermostat:
        ctx.set_thermostat(*thermostat)
    ctx.set_state(u, v)
    return ctx


def water_ctx(per_side, thermostat=None, scale=1.0):
    P = gen.SPCFW
    w = gen.water_box(per_side=per_side, seed=5)
    ctx = _lib.Context(len(w.masses), _lib.SYS_WATER, w.masses, w.charges)
    ctx.set_boundary(_lib.BC_CUBIC, [w.L, 0, 0, 0, 0, 0])
    ctx.set_kb(P["kb"])
    rc = min(0.9, 0.45 * w.L)
    ctx.add_lennard_jones(P["eps"], P["sigma"], rc)
    ctx.add_reaction_field(P["k_el"], rc, math.inf)
    ctx.set_spcfw(P["rOH"], P["aHOH"], P["kbond"], P["kangle"])
    ctx.set_precision(_lib.PREC_MIXED)
    if thermostat:
        ctx.set_thermostat(*thermostat)
    ctx.set_state(w.u, scale * w.v)
    return ctx


def expected_every(speed, dt, skin):
    """Largest M of 5, 2, 1 whose M steps, a quarter to spare, stay in the margin between the
    request and half the skin."""
    for k in (5, 2):
        if 1.25 * speed * dt * k <= 0.5 * skin * (k - 1) / (2 * k):
            return k
    return 1


@pytest.mark.parametrize("speed", [0.0, 4.0, 7.0, 40.0])
def test_interval_follows_the_largest_speed(nbx, speed):
    print(f"[case] largest speed {speed}", flush=True)
    s = gen.lj_liquid(6, rho=0.8442, T=0.01, seed=1)
    v = np.zeros_like(s.v)
    v[17] = [0.0, speed, 0.0]
    ctx = lj_ctx(s.u, v, s.L)
    ctx.vv_run(0.002, 1)
    assert ctx.stats()["build_every"] == expected_every(speed, 0.002, 0.3)
    assert {0.0: 5, 4.0: 5, 7.0: 2, 40.0: 1}[speed] == expected_every(speed, 0.002, 0.3)


def test_interval_allows_for_the_thermostat(nbx):
    # at rest, but coupled to a bath whose five-sigma speed is 5 sqrt(kb T / m)
    s = gen.lj_liquid(6, rho=0.8442, T=0.01, seed=1)
    for T, every in ((0.5, 5), (2.0, 2), (50.0, 1)):
        print(f"[case] thermostat T={T}", flush=True)
        assert expected_every(5 * math.sqrt(T), 0.002, 0.3) == every
        ctx = lj_ctx(s.u, np.zeros_like(s.v), s.L, thermostat=(_lib.THERM_LANGEVIN, T, 1.0))
        ctx.vv_run(0.002, 1)
        assert ctx.stats()["build_every"] == every


def test_interval_of_water(nbx):
    # bonds can speed up atoms that no thermostat cools
    print("[case] water, no thermostat", flush=True)
    ctx = water_ctx(8, scale=0.1)
    ctx.vv_run(0.0005, 2)
    assert ctx.stats()["build_every"] == 1
    print("[case] water, Berendsen 300 K", flush=True)
    ctx = water_ctx(8, (_lib.THERM_BERENDSEN, 300.0, 0.1))
    ctx.vv_run(0.0005, 2)
    assert ctx.stats()["build_every"] > 1


@pytest.mark.parametrize("cells,lanes", [(6, 32), (10, 32), (11, 16), (16, 16), (17, 8), (26, 4)])
def test_lanes_follow_the_size(nbx, cells, lanes):
    print(f"[case] lanes, {4 * cells ** 3} atoms", flush=True)
    s = gen.lj_liquid(cells, rho=0.8442, T=0.5, seed=cells)
    ctx = lj_ctx(s.u, s.v, s.L)
    ctx.vv_run(0.002, 1)
    assert ctx.stats()["lanes"] == lanes


def test_lanes_of_water(nbx):
    for per_side, lanes in ((11, 32), (12, 16)):   # 3,993 and 5,184 atoms
        print(f"[case] lanes, water {per_side}^3", flush=True)
        ctx = water_ctx(per_side)
        ctx.vv_run(0.0005, 1)
        assert ctx.stats()["lanes"] == lanes


def test_another_time_step_chooses_again(nbx):
    s = gen.lj_liquid(6, rho=0.8442, T=0.5, seed=3)
    speed = float(np.sqrt((s.v ** 2).sum(1)).max())
    small, large = 1e-4, 0.03 / speed   # M = 5; past M = 2
    assert expected_every(0.8 * speed, large, 0.3) == 1 and expected_every(2 * speed, small, 0.3) == 5
    print("[case] small step, then a large one", flush=True)
    ctx = lj_ctx(s.u, s.v, s.L)
    ctx.vv_run(small, 8)
    assert ctx.stats()["build_every"] == 5
    ctx.vv_run(large, 3)
    st = ctx.stats()
    assert st["build_every"] == 1 and st["stale_replays"] == 0
    print("[case] and back", flush=True)
    ctx.vv_run(small, 20)
    st = ctx.stats()
    assert st["build_every"] == 5 and st["stale_replays"] == 0


def test_another_time_step_looks_at_the_speeds_again(nbx):
    s = gen.lj_liquid(6, rho=0.8442, T=0.1, seed=3)
    ctx = lj_ctx(s.u, s.v, s.L)
    d = s.u - s.u[0]
    d -= s.L * np.rint(d / s.L)
    r = np.sqrt((d ** 2).sum(1))
    r[0] = np.inf
    s.u[r.argmin()] = s.u[0] + 0.75 * d[r.argmin()] / r.min()   # two atoms thrown apart
    ctx.set_state(s.u, 0 * s.v)
    print("[case] at rest, then moving", flush=True)
    ctx.vv_run(1e-4, 100)
    assert ctx.stats()["build_every"] == 5
    speed = float(np.sqrt((ctx.get_state()[1] ** 2).sum(1)).max())
    assert speed > 4.0
    ctx.vv_run(2e-3, 1)
    assert ctx.stats()["build_every"] == expected_every(speed, 2e-3, 0.3) < 5


def test_learned_run_keeps_its_own_request(nbx):
    """A learned run has a build opportunity at every step: the interval that a plain run
    before it chose changes neither its lists nor its steps."""
    got = []
    for plain in (False, True):
        print(f"[case] learned run, after a plain one: {plain}", flush=True)
        s = gen.lj_liquid(5, rho=0.8442, T=0.9, seed=6)
        ctx = lj_ctx(s.u, s.v, s.L)
        if plain:
            ctx.vv_run(1e-4, 0)
            assert ctx.stats()["build_every"] == 5
        m = _lib.Model(0)
        m.set(np.zeros(M.NPARAM), np.concatenate([np.zeros(35), np.ones(35), np.ones(6)]))
        rep = ctx.learned_run(m, 0.005, 4, 80, drift_tol=1.0, check_every=40)
        assert rep["strided_steps"] == 80
        got.append((rep["list_builds"], *ctx.get_state()))
    assert got[0][0] == got[1][0]
    assert np.array_equal(got[0][1], got[1][1]) and np.array_equal(got[0][2], got[1][2])


def test_replayed_blocks_hold_whole_intervals(nbx, monkeypatch):
    # blocks of 4 or 8 steps can be captured with M = 1 or 2, not with 5
    s = gen.lj_liquid(6, rho=0.8442, T=0.1, seed=1)
    for steps, every in ((4, 2), (8, 2), (50, 5), (0, 5)):
        print(f"[case] blocks of {steps} steps", flush=True)
        monkeypatch.setenv("NBX_GRAPH_STEPS", str(steps))
        ctx = lj_ctx(s.u, s.v, s.L)
        ctx.vv_run(0.002, 10)
        assert ctx.stats()["build_every"] == every
