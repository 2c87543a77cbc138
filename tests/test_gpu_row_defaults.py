"""Row passes of new plans (GPU) on both sides of the rules that pick them by
the number of rows (grid rows x slots): the default shapes of short rows at
1024 and 4096 rows, and the 2048-point complex128 pass at 256 workgroups, up to
which it keeps its coefficients in registers. One full step, real and imaginary
time, against the oracle to the parity tests' tolerances (1e-11 complex128,
2e-4 complex64)."""

import numpy as np
import pytest

from cases import ground, raman_lab
from oracle.reference_path import OraclePropagator
from spinor_gpe.engine import autotune
from spinor_gpe.engine.plan import InstanceSpec, Plan

pytestmark = pytest.mark.gpu


def _check(gpu, make, ny, nx, slots, prec, shape=None):
    ps, time, dt = make(mesh=(nx, ny))
    oracle = OraclePropagator(ps, dt, time=time)
    oracle.run(1)
    plan = Plan(gpu, prec, ny, nx, slots)
    if shape is not None:
        cur = plan.tuning()
        plan.tune(shape[0], shape[1], cur[2], cur[3])
    spec = InstanceSpec.from_spin(ps, time, dt)
    states = [plan.new_state(ps.psik) for _ in range(slots)]
    for slot, st in enumerate(states):
        plan.set_slot(slot, spec, st)
    plan.full_steps(1)
    plan.sync()
    want = np.stack(oracle.psik_numpy())
    for st in states:
        err = np.linalg.norm(st.cpu().numpy() - want) / np.linalg.norm(want)
        assert err < (1e-11 if prec == 'c128' else 2e-4), err


@pytest.mark.parametrize('prec', ['c128', 'c64'])
@pytest.mark.parametrize('make', [ground, raman_lab])
@pytest.mark.parametrize('nx', [64, 128, 256])
@pytest.mark.parametrize('ny,slots', [(64, 16), (64, 17), (128, 32), (128, 33), (2, 1)])
def test_default_rows(gpu, monkeypatch, ny, slots, nx, make, prec):
    monkeypatch.setenv('SGPE_NO_TUNE_CACHE', '1')
    print(f"[row default] {ny}x{nx} x{slots} {prec} {make.__name__}", flush=True)
    _check(gpu, make, ny, nx, slots, prec)


@pytest.mark.parametrize('make', [ground, raman_lab])
@pytest.mark.parametrize('ny,slots', [(256, 1), (128, 2), (256, 2), (512, 1)])
def test_long_rows(gpu, ny, slots, make):
    for shape in autotune.shapes(0, 'c128', 2048):
        if shape[0] != 8:
            continue
        print(f"[long row] {ny}x2048 x{slots} {shape} {make.__name__}", flush=True)
        _check(gpu, make, ny, 2048, slots, 'c128', shape)
