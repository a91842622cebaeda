"""The FP64 pair kernel and the fused step against the oracle, bit for bit: sizes around a
wavefront, sources filtered by box fractions and not, every law and boundary condition,
several potentials, thermostats, saved frames, split runs."""
import math

import numpy as np
import pytest

import oracle_lib as O
from nbodysimulator import _lib
from nbodysimulator import generators as gen

pytestmark = pytest.mark.gpu

LAWS = {"lj": [("lj", 1.0, 1.0, 2.5)], "coulomb": [("el", 1.3, 2.2)], "open": [("el", 1.3, math.inf)],
        "rf": [("rf", 1.3, 2.2, 78.5)], "gravity": [("grav", 0.7)],
        "lj+rf": [("lj", 1.0, 1.0, 2.5), ("rf", 1.3, 2.2, math.inf)],
        "grav+el+lj": [("grav", 0.7), ("el", 1.3, math.inf), ("lj", 1.0, 1.0, 2.5)]}
ADD = {"lj": ("add_lennard_jones", O.TERM_LJ), "el": ("add_electrostatic", O.TERM_ELEC),
       "rf": ("add_reaction_field", O.TERM_RF), "grav": ("add_gravitational", O.TERM_GRAV)}


def pair(n, law, bc, L, seed=0, therm=None):
    rng = np.random.default_rng([n, seed])
    m, q = rng.uniform(0.5, 2.0, n), rng.uniform(-0.4, 0.4, n)
    box = {"cubic": [L, 0, 0, 0, 0, 0], "lohi": [0, L, -L / 2, L / 2, 0, 1.1 * L], "infinite": None}[bc]
    kind = {"cubic": _lib.BC_CUBIC, "lohi": _lib.BC_PERIODIC, "infinite": _lib.BC_INFINITE}[bc]
    ctx = _lib.Context(n, _lib.SYS_POTENTIAL, m, q)
    ctx.set_boundary(kind, box)
    ctx.set_kb(1.0)
    orc = O.System(m, charges=q, bc=O.make_bc(kind, L if bc == "cubic" else box))
    for name, *p in LAWS[law]:
        getattr(ctx, ADD[name][0])(*p)
        orc.add(ADD[name][1], *p)
    if therm:
        ctx.set_thermostat(*therm)
        orc.thermostat(*therm)
    return ctx, orc, rng


def lattice(n, L, rng):
    c = math.ceil(n ** (1.0 / 3.0) - 1e-9)
    g = np.stack(np.meshgrid(*[np.arange(c)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    return np.ascontiguousarray((g + 0.5) * (L / c) + 0.03 * rng.standard_normal((n, 3)))


@pytest.mark.parametrize("bc", ["cubic", "lohi", "infinite"])
@pytest.mark.parametrize("law", list(LAWS))
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 200, 513])
def test_forces_bitwise(nbx, n, law, bc):
    print(f"[case] fp64 pairs n={n} law={law} bc={bc}", flush=True)
    # the smallest boxes hold the cutoff more than half (no filter), the larger ones filter
    L = 1.2 * max(n, 8) ** (1.0 / 3.0)
    ctx, orc, rng = pair(n, law, bc, L)
    u = lattice(n, L, rng)
    u[::5] += L * rng.integers(-40, 41, (len(u[::5]), 3))      # unwrapped, many boxes away
    assert np.array_equal(ctx.rhs(u), orc.rhs(u))


def test_forces_of_coordinates_past_the_filter_margin(nbx):
    print("[case] fp64 pairs, coordinates 2^21 boxes away", flush=True)
    n, L = 300, 8.0
    ctx, orc, rng = pair(n, "lj", "cubic", L)
    u = lattice(n, L, rng)
    u[7] += 2.0 ** 21 * L
    u[100:110] -= 3.0 * 2.0 ** 21 * L
    assert np.array_equal(ctx.rhs(u), orc.rhs(u))


@pytest.mark.parametrize("therm", [None, (_lib.THERM_BERENDSEN, 1.2, 0.05),
                                   (_lib.THERM_ANDERSEN, 1.1, 5.0), (_lib.THERM_LANGEVIN, 1.3, 1.0),
                                   (_lib.THERM_NOSEHOOVER, 1.2, 0.3)])
@pytest.mark.parametrize("law,bc,n", [("lj", "cubic", 300), ("lj+rf", "cubic", 130),
                                      ("grav+el+lj", "infinite", 65), ("gravity", "infinite", 70),
                                      ("lj", "lohi", 64)])
def test_runs_match_oracle(nbx, law, bc, n, therm):
    print(f"[case] fp64 runs n={n} law={law} bc={bc} therm={therm}", flush=True)
    L = 1.2 * n ** (1.0 / 3.0)
    ctx, orc, rng = pair(n, law, bc, L, 1, therm)
    u, v = lattice(n, L, rng), rng.standard_normal((n, 3))
    ctx.set_state(u, v)
    uf, vf = ctx.vv_run(0.002, 21, seed=9, save_every=4)
    ctx.vv_run(0.002, 1, seed=9)
    ctx.vv_run(0.002, 12, seed=9)
    u1, v1 = ctx.get_state()
    uo, vo, (ufo, vfo) = orc.vv_run(u, v, 0.002, 34, seed=9, save_every=4)
    assert uf.shape[0] == 6 and ctx.steps_taken() == 34
    if therm is None or therm[0] in (_lib.THERM_BERENDSEN, _lib.THERM_NOSEHOOVER):
        if therm is None or therm[0] == _lib.THERM_BERENDSEN:   # zeta restarts with a new run
            assert np.array_equal(u1, uo) and np.array_equal(v1, vo)
        assert np.array_equal(uf, ufo[:6]) and np.array_equal(vf, vfo[:6])
    else:   # logarithm and cosine of the noise: libm
        for a, b in ((u1, uo), (v1, vo), (uf, ufo[:6]), (vf, vfo[:6])):
            assert np.abs(a - b).max() <= 1e-11 * np.abs(b).max()


@pytest.mark.parametrize("therm", [None, (_lib.THERM_BERENDSEN, 300.0, 0.1),
                                   (_lib.THERM_ANDERSEN, 300.0, 50.0),
                                   (_lib.THERM_LANGEVIN, 300.0, 5.0)])
@pytest.mark.parametrize("el,rc", [("coulomb", 0.35), ("rf", 0.35), ("coulomb", 0.9)])
def test_water_runs_match_oracle(nbx, el, rc, therm):
    print(f"[case] fp64 water el={el} rc={rc} therm={therm}", flush=True)
    w, P = gen.water_box(4, seed=3), gen.SPCFW
    n = len(w.masses)
    ctx = _lib.Context(n, _lib.SYS_WATER, w.masses, w.charges)
    ctx.set_boundary(_lib.BC_CUBIC, [w.L, 0, 0, 0, 0, 0])
    ctx.set_kb(P["kb"])
    ctx.add_lennard_jones(P["eps"], P["sigma"], rc)
    elec = (P["k_el"], rc) if el == "coulomb" else (P["k_el"], rc, math.inf)
    (ctx.add_electrostatic if el == "coulomb" else ctx.add_reaction_field)(*elec)
    ctx.set_spcfw(P["rOH"], P["aHOH"], P["kbond"], P["kangle"])
    orc = O.System(w.masses, charges=w.charges, water=True, bc=O.make_bc(O.BC_CUBIC, w.L), kb=P["kb"])
    orc.water_params((P["eps"], P["sigma"], rc), O.TERM_ELEC if el == "coulomb" else O.TERM_RF, elec,
                     P["rOH"], P["aHOH"], P["kbond"], P["kangle"])
    if therm:
        ctx.set_thermostat(*therm)
        orc.thermostat(*therm)
    ctx.set_state(w.u, w.v)
    uf, vf = ctx.vv_run(0.0005, 15, seed=5, save_every=5)
    u, v = ctx.get_state()
    uo, vo, (ufo, vfo) = orc.vv_run(w.u, w.v, 0.0005, 15, seed=5, save_every=5)
    for a, b in ((u, uo), (v, vo), (uf, ufo), (vf, vfo)):      # acos in the angle: libm
        assert np.abs(a - b).max() <= 1e-11 * np.abs(b).max()


@pytest.mark.parametrize("law,bc", [("gravity", "infinite"), ("open", "infinite"), ("lj", "cubic"),
                                    ("rf", "cubic"), ("lj", "lohi"), ("grav+el+lj", "infinite"),
                                    ("magnetic", "infinite")])
@pytest.mark.parametrize("n", [1, 2, 3, 8, 9, 21, 33, 47, 48, 49])
def test_small_runs_bitwise(nbx, n, law, bc):
    print(f"[case] fp64 small run n={n} law={law} bc={bc}", flush=True)
    L = 1.2 * max(n, 8) ** (1.0 / 3.0)
    if law == "magnetic":
        rng = np.random.default_rng(n)
        m, mm = rng.uniform(0.5, 2.0, n), 0.1 * rng.standard_normal((n, 3))
        ctx, orc = _lib.Context(n, _lib.SYS_POTENTIAL, m), O.System(m).moments(mm)
        ctx.set_moments(mm)
        ctx.add_magnetostatic(0.3)
        orc.add(O.TERM_MAG, 0.3)
    else:
        ctx, orc, rng = pair(n, law, bc, L, 2)
    u, v = lattice(n, L, rng), 0.3 * rng.standard_normal((n, 3))
    ctx.set_state(u, v)
    uf, vf = ctx.vv_run(0.002, 25, save_every=3)
    ctx.vv_run(0.002, 1)
    ctx.vv_run(0.002, 14)
    u1, v1 = ctx.get_state()
    uo, vo, (ufo, vfo) = orc.vv_run(u, v, 0.002, 40, save_every=3)
    assert np.array_equal(u1, uo) and np.array_equal(v1, vo) and ctx.steps_taken() == 40
    assert np.array_equal(uf, ufo[:9]) and np.array_equal(vf, vfo[:9])


def test_small_run_of_several_launches(nbx):
    print("[case] fp64 small run, 45,000 steps", flush=True)
    ctx, orc, rng = pair(2, "gravity", "infinite", 3.0)
    u, v = np.array([[0.0, 0, 0], [1.0, 0, 0]]), np.array([[0.0, -0.3, 0], [0, 0.6, 0.1]])
    ctx.set_state(u, v)
    uf, vf = ctx.vv_run(1e-3, 45000, save_every=7)
    uo, vo, (ufo, vfo) = orc.vv_run(u, v, 1e-3, 45000, save_every=7)
    assert np.array_equal(uf, ufo) and np.array_equal(vf, vfo)
    assert np.array_equal(ctx.get_state()[0], uo)


# Four wavefronts per target up to 1,536 targets, in rounds of at most 1,024 sources: a round's
# edge, the last targets of the rule and the first past it, and a cutoff of nearly half the
# box, with about half of a wavefront's 256 sources in range
@pytest.mark.parametrize("law", ["lj", "rf", "wide"])
@pytest.mark.parametrize("n", [255, 257, 1024, 1025, 1536, 1537, 2049])
def test_forces_by_four_wavefronts_bitwise(nbx, monkeypatch, n, law):
    print(f"[case] fp64 pairs by four wavefronts n={n} law={law}", flush=True)
    L = 1.2 * n ** (1.0 / 3.0)
    monkeypatch.setitem(LAWS, "wide", [("el", 1.3, 0.49 * L)])
    ctx, orc, rng = pair(n, law, "cubic", L)
    u = lattice(n, L, rng)
    u[::5] += L * rng.integers(-40, 41, (len(u[::5]), 3))
    assert np.array_equal(ctx.rhs(u), orc.rhs(u))
    v = rng.standard_normal((n, 3))
    ctx.set_state(u, v)
    ctx.vv_run(0.001, 2)
    uo, vo, _ = orc.vv_run(u, v, 0.001, 2)
    u1, v1 = ctx.get_state()
    assert np.array_equal(u1, uo) and np.array_equal(v1, vo)
