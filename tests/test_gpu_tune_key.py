"""Kept tuning results name the revision of the kernels that they were timed on."""
import numpy as np
import pytest

from nbodysimulator import _lib
from nbodysimulator import generators as gen

pytestmark = pytest.mark.gpu

ARCH = "arch=gfx950"


def test_a_shape_of_replaced_kernels_is_not_applied(nbx, tmp_path, monkeypatch):
    print("[case] tuning results without a kernel revision", flush=True)
    # lines as they were written before results named it
    old = tmp_path / "tune.tsv"
    grav = f"gravity n=1000 L=0 rc=0 dt=0.001 trial=21 sys=0 therm=0 lj=0 el=0 {ARCH}"
    s = gen.lj_liquid(5, rho=0.8442, T=0.8, seed=3)
    lst = f"list n=500 L={s.L:.17g} rc=2.5 dt=0.0050000000000000001 trial=21 sys=0 therm=0 lj=1 el=0 {ARCH}"
    old.write_text(f"{grav}\t1\t64\t0.01\t0.02\t1\n{lst}\t4\t0.75\t0.01\t0.02\t1\n")
    monkeypatch.setenv("NBX_TUNE_CACHE", str(old))
    u, v, m = gen.plummer(1000, seed=4)
    g = _lib.Context(1000, _lib.SYS_POTENTIAL, m)
    g.add_gravitational(1.0)
    g.set_precision(_lib.PREC_MIXED)
    g.set_state(u, v)
    assert g.autotune(0.001, 21)["candidates"] > 0
    ctx = _lib.Context(500, _lib.SYS_POTENTIAL, np.ones(500))
    ctx.set_boundary(_lib.BC_CUBIC, [s.L, 0, 0, 0, 0, 0])
    ctx.add_lennard_jones(1.0, 1.0, 2.5)
    ctx.set_kb(1.0)
    ctx.set_precision(_lib.PREC_MIXED)
    ctx.set_state(s.u, s.v)
    assert ctx.autotune(0.005, 21)["candidates"] > 0
    # the results of these trials were appended under the present revision and are found again
    assert len(old.read_text().splitlines()) == 4
    assert g.autotune(0.001, 21)["candidates"] == 0
    assert ctx.autotune(0.005, 21)["candidates"] == 0
