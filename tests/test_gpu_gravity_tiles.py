"""The tiled gravity kernel at the edges of its tiles: every size class (64, 128 and 256
bodies per narrow tile up to 32,768 bodies, 1,024 per wide tile, rings of one launch and of several), partial
last tiles, odd and even rings, equal and unequal masses."""
import numpy as np
import pytest

import oracle_lib as O
from nbodysimulator import _lib
from nbodysimulator import generators as gen

pytestmark = pytest.mark.gpu


def mixed_accel(m, u):
    ctx = _lib.Context(len(m), _lib.SYS_POTENTIAL, m)
    ctx.add_gravitational(1.0)
    ctx.set_precision(_lib.PREC_MIXED)
    ctx.set_state(u, np.zeros_like(u))
    dt = 2.0 ** -60     # one step from rest: a = (v1 - v0) / dt
    _, vf = ctx.vv_run(dt, 1, save_every=1)
    return (vf[1] - vf[0]) / dt


# FP32 pair forces from positions rounded to FP32: the bar of the engine's gravity tests at
# full size, 5e-5 of the largest force
@pytest.mark.parametrize("equal", [True, False])
@pytest.mark.parametrize("n", [1, 2, 3, 63, 64, 65, 127, 129, 200, 1000, 3001, 4096, 4097, 6000,
                               8192, 8193, 12345, 16384, 16385, 17409, 32768, 32769, 33000, 140001])
def test_every_pair_once(nbx, n, equal):
    print(f"[case] gravity tiles n={n} equal={equal}", flush=True)
    u, _, m = gen.plummer(n, seed=n)
    rng = np.random.default_rng(n)
    if not equal:
        m = m * rng.uniform(0.5, 2.0, n)
    a = mixed_accel(m, u)
    # first, last and random targets (all of them for small systems)
    pick = np.arange(n) if n <= 1000 else np.unique(np.concatenate(
        [[0, 63, 64, 1023, 1024, n // 2, n - 65, n - 1], rng.choice(n, 56, replace=False)]))
    ref = np.zeros((len(pick), 3))
    lib = O.load()
    for k, i in enumerate(pick):
        lib.orc_grav_accel(O.dp(ref[k]), O.dp(np.ascontiguousarray(u)), int(i), n, O.dp(m), 1.0)
    if n == 1:
        assert np.array_equal(a, np.zeros((1, 3)))
        return
    scale = np.abs(ref).max()
    assert np.abs(a[pick] - ref).max() <= 5e-5 * scale
    # every pair enters both bodies: the total momentum stays at rest
    f = (m[:, None] * a)
    assert np.abs(f.sum(axis=0)).max() <= 1e-5 * np.abs(f).sum()


def test_autotuner_times_the_steps_not_their_launches(nbx):
    # a step takes at least its force kernel; half of it leaves room for the clock
    print("[case] gravity autotuner n=40000", flush=True)
    n = 40000
    u, v, m = gen.plummer(n, seed=3)
    ctx = _lib.Context(n, _lib.SYS_POTENTIAL, m)
    ctx.add_gravitational(1.0)
    ctx.set_precision(_lib.PREC_MIXED)
    ctx.set_state(u, v)
    tuned = ctx.autotune(1e-3, 10)
    ctx.set_state(u, v)
    kernel_ms, _ = ctx.time_force_kernel(5)
    assert tuned["entry_ms_per_step"] >= 0.5 * kernel_ms
