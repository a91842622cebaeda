"""The radial distribution histogram at the edges of its tiles, block sizes and histogram
placements: every count equals the oracle's."""
import numpy as np
import pytest

import oracle_lib as O
from nbodysimulator import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nframes,maxbin", [
    (1, 2, 10), (2, 1, 1), (63, 1, 50), (64, 3, 1000), (65, 1, 7), (130, 2, 8000), (130, 2, 8001),
    (700, 2, 1000), (700, 3, 20000), (1500, 3, 333), (3000, 4, 1000)])
def test_counts_equal_the_oracle(nbx, n, nframes, maxbin):
    print(f"[case] rdf n={n} frames={nframes} maxbin={maxbin}", flush=True)
    rng = np.random.default_rng(n + maxbin)
    L = 0.9 * n ** (1.0 / 3.0) + 1.0
    frames = rng.uniform(0, L, (nframes, n, 3))
    frames[-1, ::3] += L * rng.integers(-3, 4, (len(frames[-1, ::3]), 3))   # boxes away
    ctx = _lib.Context(n, _lib.SYS_POTENTIAL, np.ones(n))
    ctx.set_boundary(_lib.BC_CUBIC, [L, 0, 0, 0, 0, 0])
    rs, gr = ctx.rdf(frames, maxbin)
    rso, gro = O.rdf(frames, L, maxbin=maxbin)
    assert np.array_equal(rs, rso) and np.array_equal(gr, gro)
    if maxbin <= _lib.RDF_NOALLOC_MAXBIN:
        assert np.array_equal(ctx.rdf_noalloc(frames, maxbin)[1], gro)


def test_water_counts_oxygens(nbx):
    print("[case] rdf water", flush=True)
    rng = np.random.default_rng(4)
    n, L = 3 * 150, 3.0
    frames = rng.uniform(-L, 2 * L, (2, n, 3))
    ctx = _lib.Context(n, _lib.SYS_WATER, np.tile([16.0, 1.0, 1.0], n // 3), np.tile([-.8, .4, .4], n // 3))
    ctx.set_boundary(_lib.BC_CUBIC, [L, 0, 0, 0, 0, 0])
    gr = ctx.rdf(frames, 200)[1]
    assert np.array_equal(gr, O.rdf(frames, L, indxs=np.arange(0, n, 3), maxbin=200)[1])


@pytest.mark.parametrize("L,maxbin", [(8.0, 64), (8.0, 1000), (7.3, 73), (7.3, 4001)])
def test_distances_on_bin_edges_and_far_images(nbx, L, maxbin):
    # distances that are whole multiples of a bin or of half the box, whose bin only the FP64
    # square root and division decide, and atoms too far away for the FP32 estimate
    print(f"[case] rdf edges L={L} maxbin={maxbin}", flush=True)
    rng = np.random.default_rng(maxbin)
    n = 300
    grid = rng.integers(0, 16, (n, 3)) * (L / 16)            # on multiples of L / 16
    line = np.zeros((n, 3))
    line[:, 0] = rng.integers(0, maxbin, n) * (L / maxbin)   # on bin edges along x
    far = rng.uniform(0, L, (n, 3))
    far[::7] += L * 2000
    far[1::7] -= L * 1023.5
    frames = np.stack([grid, line, far])
    ctx = _lib.Context(n, _lib.SYS_POTENTIAL, np.ones(n))
    ctx.set_boundary(_lib.BC_CUBIC, [L, 0, 0, 0, 0, 0])
    assert np.array_equal(ctx.rdf(frames, maxbin)[1], O.rdf(frames, L, maxbin=maxbin)[1])
