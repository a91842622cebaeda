"""Energies over tiles of pairs and ordered sums, at the edges of the tiles and chunks: every
boundary condition, Lennard-Jones with Coulomb or a reaction field, kinetic energy and
temperature bit for bit."""
import math

import numpy as np
import pytest

import oracle_lib as O
from nbodysimulator import _lib

pytestmark = pytest.mark.gpu

BCS = {"cubic": (_lib.BC_CUBIC, lambda L: [L, 0, 0, 0, 0, 0], lambda L: O.make_bc(O.BC_CUBIC, L)),
       "infinite": (_lib.BC_INFINITE, lambda L: None, lambda L: O.make_bc(O.BC_INFINITE))}


# Pair terms summed in another order than the oracle's single running sum: n^2 / 2 terms, each
# sum within 1e-12 of its value where the close pairs of a random gas dominate (no
# cancellation), the bar of the engine's Lennard-Jones energy tests
@pytest.mark.parametrize("bc", ["cubic", "infinite"])
@pytest.mark.parametrize("el", ["none", "coulomb", "open", "rf"])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 129, 1024, 1025, 1500])
def test_energies_match_oracle(nbx, n, el, bc):
    print(f"[case] energies n={n} el={el} bc={bc}", flush=True)
    rng = np.random.default_rng(n)
    L = n ** (1.0 / 3.0) + 2.0
    u, v = rng.uniform(-L, 2 * L, (n, 3)), rng.standard_normal((n, 3))
    m, q = rng.uniform(0.5, 2.0, n), rng.uniform(0.1, 0.4, n)
    kind, box, obc = BCS[bc]
    ctx = _lib.Context(n, _lib.SYS_POTENTIAL, m, q)
    ctx.set_boundary(kind, box(L))
    ctx.set_kb(1.0)
    orc = O.System(m, charges=q, bc=obc(L))
    R = 0.4 * L
    if el == "coulomb":
        ctx.add_electrostatic(1.3, R)
        orc.add(O.TERM_ELEC, 1.3, R)
    elif el == "open":
        ctx.add_electrostatic(1.3, math.inf)
        orc.add(O.TERM_ELEC, 1.3, math.inf)
    elif el == "rf":
        ctx.add_reaction_field(1.3, R, 78.5)
        orc.add(O.TERM_RF, 1.3, R, 78.5)
    ctx.add_lennard_jones(1.0, 1.0, 2.5)
    orc.add(O.TERM_LJ, 1.0, 1.0, 2.5)
    ctx.set_state(u, v)
    ke, pe, pg = ctx.energies()
    assert ke == orc.kinetic_energy(v) and pg == 0.0
    assert pe == pytest.approx(orc.potential_energy(u), rel=1e-11, abs=1e-300)
    assert ctx.temperature() == O.load().orc_md_temperature(O.dp(v), O.dp(m), 1.0, n, 0)


@pytest.mark.parametrize("shift", [1000, 3000])
def test_energies_with_atoms_many_boxes_away(nbx, shift):
    # on either side of the distance up to which pairs are found in FP32; the images differ
    # from the atoms in the box by the rounding of shift * L only (1e-12 of a distance, 1e-11
    # of a close pair's energy)
    print(f"[case] energies, atoms {shift} boxes away", flush=True)
    n = 1025
    rng = np.random.default_rng(shift)
    L = 16.0   # shift * L is exact
    g = np.stack(np.meshgrid(*[np.arange(11)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    u = g * (L / 11) + rng.uniform(0, 0.3, (n, 3))
    w = u.copy()
    w[::50] += shift * L * rng.integers(-1, 2, w[::50].shape)
    pes = []
    for x in (u, w):
        ctx = _lib.Context(n, _lib.SYS_POTENTIAL, np.ones(n))
        ctx.set_boundary(_lib.BC_CUBIC, [L, 0, 0, 0, 0, 0])
        ctx.add_lennard_jones(1.0, 1.0, 2.5)
        ctx.set_state(x, np.zeros_like(x))
        pes.append(ctx.energies()[1])
    orc = O.System(np.ones(n), bc=O.make_bc(O.BC_CUBIC, L)).add(O.TERM_LJ, 1.0, 1.0, 2.5)
    assert pes[0] == pytest.approx(orc.potential_energy(u), rel=1e-11)
    assert pes[1] == pytest.approx(orc.potential_energy(w), rel=1e-11)
    assert pes[1] == pytest.approx(pes[0], rel=1e-9)
