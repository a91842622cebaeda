"""Lists that go stale between two build opportunities at the interval that the run chose by
itself: the state allows five steps, and a few steps later atoms outrun it."""
import numpy as np
import pytest

from nbodysimulator import _lib
from nbodysimulator import generators as gen
from test_gpu_build_rule import defaults, lj_ctx, water_ctx  # noqa: F401

pytestmark = pytest.mark.gpu

# a bath at 20 K allows M = 5; the molecules, placed at random angles, fall together
COLD_BATH = (_lib.THERM_BERENDSEN, 20.0, 10.0)


def colliding(cells, distance):
    """A cold liquid in which the first atom's neighbour has been pushed towards it."""
    s = gen.lj_liquid(cells, rho=0.8442, T=0.3, seed=cells + 40, jitter=0.03)
    d = s.u - s.u[0]
    d -= s.L * np.rint(d / s.L)
    r = np.sqrt((d ** 2).sum(1))
    r[0] = np.inf
    j = int(r.argmin())
    s.u[j] = s.u[0] + d[j] * (distance / r[j])
    return s


@pytest.mark.parametrize("every", [None, 5])
def test_stale_half_cell_bins_are_no_overflow(nbx, monkeypatch, every):
    """Bins made by the builds: an atom past 3/4 skin counts as an overflow.  Where the list
    went stale first, larger lists are no remedy, and the run does not end for want of room."""
    if every:
        monkeypatch.setenv("NBX_BUILD_EVERY", str(every))
    print(f"[case] colliding atoms, half-size cells, build every {every}", flush=True)
    s = colliding(14, 0.7)
    ctx = lj_ctx(s.u, s.v, s.L, R=5.0, skin=0.2)
    ctx.vv_run(0.002, 40)
    assert ctx.stats()["cells_per_side"] == 8 and ctx.stats()["stale_replays"] == 1
    print(f"[case] water at rest, half-size cells, build every {every}", flush=True)
    ctx = water_ctx(13, COLD_BATH, scale=0.0)
    ctx.vv_run(0.001, 100)
    assert ctx.stats()["cells_per_side"] == 6 and ctx.stats()["stale_replays"] == 1


LAYOUTS = [
    (4, 2.5),     # no cells: 256 atoms, all pairs
    (6, 2.5),     # bins made once, 3 cells per side
    (10, 2.5),    # bins of each build's step
    (13, 2.5),    # the same, the state sorted by cell
    (14, 5.0),    # half-size cells binned by the builds
]


@pytest.mark.parametrize("distance", [0.7, 0.75])   # stale after 5 steps, and later
@pytest.mark.parametrize("cells,R", LAYOUTS)
def test_stale_lists_leave_no_trace_of_how_steps_were_run(nbx, monkeypatch, cells, R, distance):
    """The trajectory depends on the state, the time step and the configuration alone -- not on
    a run before it on the same context, on where runs are split or on the frames saved."""
    print(f"[case] stale lists, cells={cells} R={R} distance={distance}", flush=True)
    s = colliding(cells, distance)
    if cells == 13:   # a state that the run re-sorts
        p = np.random.default_rng(7).permutation(len(s.u))
        s.u, s.v = s.u[p], s.v[p]
        monkeypatch.setenv("NBX_SORT_EVERY", "50")
    dt, steps = 0.002, 160

    def after(ctx, parts):
        for k in parts:
            ctx.vv_run(dt, k)
        return ctx.get_state()

    def fresh():
        return lj_ctx(s.u, s.v, s.L, R, skin=0.2)

    ctx = fresh()
    ua, va = after(ctx, [steps])
    st = ctx.stats()
    assert st["stale_replays"] == 1 and st["build_every"] == 1
    print("[case]   the same calls again", flush=True)
    ctx.set_state(s.u, s.v)
    ub, vb = after(ctx, [steps])
    assert np.array_equal(ua, ub) and np.array_equal(va, vb)
    assert ctx.stats()["stale_replays"] == 1
    for parts in ([4, 156], [1] * 12 + [148], [53, 107]):
        print(f"[case]   split {parts[:2]}", flush=True)
        c = fresh()
        ub, vb = after(c, parts)
        assert np.array_equal(ua, ub) and np.array_equal(va, vb)
        assert c.stats()["stale_replays"] == 1
    print("[case]   frames", flush=True)
    uf, vf = fresh().vv_run(dt, steps, save_every=4)
    assert np.array_equal(ua, uf[-1]) and np.array_equal(va, vf[-1])
    print("[case]   blocks of 20 steps", flush=True)
    monkeypatch.setenv("NBX_GRAPH_STEPS", "20")
    ub, vb = after(fresh(), [steps])
    assert np.array_equal(ua, ub) and np.array_equal(va, vb)


@pytest.mark.parametrize("cells,R", LAYOUTS)
def test_stale_lists_miss_no_pair(nbx, cells, R):
    """The run that went stale against the FP64 path over the steps of the collision: a pair
    missing from a list moves atoms by 1e-3."""
    print(f"[case] stale lists against FP64, cells={cells} R={R}", flush=True)
    s = colliding(cells, 0.7)
    ctx = lj_ctx(s.u, s.v, s.L, R, skin=0.2)
    ctx.vv_run(0.002, 40)
    assert ctx.stats()["stale_replays"] == 1
    ref = lj_ctx(s.u, s.v, s.L, R)
    ref.set_precision(_lib.PREC_FP64_REF)
    ref.vv_run(0.002, 40)
    assert float(np.abs(ctx.get_state()[0] - ref.get_state()[0]).max()) < 1e-4


def test_stale_lists_of_water_with_a_thermostat(nbx):
    print("[case] stale lists, water", flush=True)
    dt = 0.0005

    def after(parts):
        c = water_ctx(13, COLD_BATH, scale=0.0)   # half-size cells binned by the builds
        for k in parts:
            c.vv_run(dt, k)
        assert c.stats()["stale_replays"] == 1
        return c.get_state()

    ua, va = after([150])
    ub, vb = after([3, 50, 97])
    assert np.array_equal(ua, ub) and np.array_equal(va, vb)


@pytest.mark.parametrize("kind", ["langevin", "andersen", "nosehoover", "euler-maruyama"])
def test_stale_lists_with_thermostats(nbx, kind):
    """The replay draws the same numbers and takes the thermostat's state back."""
    print(f"[case] stale lists, {kind}", flush=True)
    s = colliding(6, 0.7)
    therm = {"langevin": (_lib.THERM_LANGEVIN, 0.2, 1.0), "andersen": (_lib.THERM_ANDERSEN, 0.2, 5.0),
             "nosehoover": (_lib.THERM_NOSEHOOVER, 0.2, 0.5),
             "euler-maruyama": (_lib.THERM_LANGEVIN, 0.2, 1.0)}[kind]

    def after(parts):
        c = lj_ctx(s.u, s.v, s.L, skin=0.2, thermostat=therm)
        for k in parts:
            (c.em_run if kind == "euler-maruyama" else c.vv_run)(0.002, k, seed=9)
        assert c.stats()["stale_replays"] == 1
        return (*c.get_state(), c.thermostat_state())

    (ua, va, ta), (ub, vb, tb) = after([80]), after([4, 76])
    if kind == "nosehoover":
        # the drift redone at a run's start adds the temperature of the atoms in another order:
        # sqrt(3 n) roundings of 2^-53 in T, in a rate of T / tau^2 over 76 steps
        assert np.abs(ua - ub).max() < 1e-12 and np.abs(va - vb).max() < 1e-11
        assert np.allclose(ta, tb, rtol=1e-11, atol=1e-12)
    else:
        assert np.array_equal(ua, ub) and np.array_equal(va, vb)
