"""The list build's layouts: three cells per side (integer minimum images), small cells of
each step's bins, cells of more than 768 atoms, half-size cells of the previous build's bins,
and 32-bit list entries.  Every pair in range has to be in the lists exactly once, at the
start and after a run that rebuilt them, counted against a k-d tree."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

from nbodysimulator import _lib
from nbodysimulator import generators as gen

pytestmark = pytest.mark.gpu


def pairs_within(u, L, r):
    t = cKDTree(np.mod(u, L), boxsize=L)
    return int(t.count_neighbors(t, r)) - len(u)   # ordered, without the atoms themselves


@pytest.mark.parametrize("cells,rho,R,skin", [
    (2, 0.8442, 1.5, 0.3),     # all pairs, fewer atoms than lanes
    (4, 0.8442, 2.5, 0.3),     # all pairs, 256 atoms
    (5, 0.8442, 2.7, 0.3),     # all pairs, 500
    (6, 0.8442, 2.5, 0.3),     # 3 cells per side
    (8, 0.8442, 2.5, 0.3),     # 4
    (9, 0.8442, 2.5, 0.2),     # 5
    (19, 1.0, 3.6, 3.6),       # 4 of about 430 atoms: several batches, own atoms in four passes
    (14, 0.8442, 4.5, 0.3),    # half-size cells, 8 per side
    (26, 0.8442, 2.5, 0.3),    # 70,304 atoms: 32-bit entries
])
def test_lists_hold_every_pair_once(nbx, cells, rho, R, skin):
    print(f"[case] list build cells={cells} rho={rho} R={R} skin={skin}", flush=True)
    s = gen.lj_liquid(cells, rho=rho, T=0.9, seed=cells, jitter=0.03)
    # atoms in other images of the box
    u = s.u + s.L * np.random.default_rng(cells).integers(-2, 3, s.u.shape)
    ctx = _lib.Context(len(u), _lib.SYS_POTENTIAL, s.masses)
    ctx.set_boundary(_lib.BC_CUBIC, [s.L, 0, 0, 0, 0, 0])
    ctx.add_lennard_jones(1.0, 1.0, R)
    ctx.set_kb(1.0)
    ctx.set_precision(_lib.PREC_MIXED)
    ctx.set_skin(skin)
    ctx.set_state(u, s.v)
    for steps in (0, 40):
        if steps:
            ctx.vv_run(0.004, steps)
        x, _ = ctx.get_state()
        # pairs whose FP32 distance may fall on either side of the cutoff are left open: the
        # rounding of three differences and their squares, 2^-22 of the distance
        lo, hi = (pairs_within(x, s.L, R * (1 + e)) for e in (-2.4e-7, 2.4e-7))
        assert lo <= ctx.count_pairs() <= hi
