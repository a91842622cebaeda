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
