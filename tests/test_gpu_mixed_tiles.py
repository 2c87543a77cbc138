"""Mixed-radix split steps with more than one row, and wider columns, per
workgroup (GPU), as plans of many slots take them, and transforms of four
stages: rows in twos and fours, columns in tiles of 8, 13, 15 and 16, two and
three stages; different physics in neighbouring slots (real and imaginary
time, tables and dense arrays). Every slot against its own oracle run to the
parity tests' tolerances (1e-11 complex128, 2e-4 complex64)."""

import functools

import numpy as np
import pytest

import cases
from oracle.reference_path import OraclePropagator
from spinor_gpe.engine.plan import InstanceSpec, Plan

pytestmark = pytest.mark.gpu


def _runs(makers, mesh):
    out = []
    for i, make in enumerate(makers):
        ps, time, dt = make(name=f'mt{i}', mesh=mesh, seed=40 + i)
        oracle = OraclePropagator(ps, dt, time=time)
        oracle.full_step()
        oracle.single_step(oracle.dt_in, oracle.eng_in)
        out.append((ps, InstanceSpec.from_spin(ps, time, dt), np.stack(oracle.psik_numpy())))
    return out


def _check(gpu, runs, nx, ny, slots, precision):
    plan = Plan(gpu, precision, ny, nx, slots)
    states = []
    for slot in range(slots):
        ps, spec, _ = runs[slot % len(runs)]
        states.append(plan.new_state(ps.psik))
        plan.set_slot(slot, spec, states[-1])
    plan.full_steps(1)
    plan.single_step(1)
    plan.sync()
    for slot, st in enumerate(states):
        want = runs[slot % len(runs)][2]
        err = float(np.linalg.norm(st.cpu().numpy() - want) / np.linalg.norm(want))
        assert err < (1e-11 if precision == 'c128' else 2e-4), (slot, err)


# (nx, ny, slots): rows per workgroup and columns per tile on 256 CUs
SIZES = [(96, 100, 24),   # 4 rows; 8 columns
         (96, 100, 48),   # 4 rows; 8 columns (complex128), 16 (complex64)
         (208, 286, 16),  # 2 rows of three stages; 8 and 13 columns of three stages
         (600, 66, 16)]   # 2 rows of three stages; columns of two stages in tiles of 8 and 15


@pytest.mark.parametrize('precision', ['c128', 'c64'])
@pytest.mark.parametrize('dense', [False, True])
@pytest.mark.parametrize('size', SIZES, ids=str)
def test_many_slots(gpu, size, dense, precision):
    nx, ny, slots = size
    print(f"[mixed tiles] {nx}x{ny} x{slots} dense={dense} {precision}", flush=True)
    makers = [cases.ground, cases.raman_lab, cases.raman_rot] + ([cases.dense_ops, cases.dense_kin] if dense else [])
    _check(gpu, _runs(makers, (nx, ny)), nx, ny, slots, precision)


@pytest.mark.parametrize('precision', ['c128', 'c64'])
@pytest.mark.parametrize('size', [(1250, 64), (64, 1250), (36, 2000), (2000, 36)], ids=str)
@pytest.mark.parametrize('make', [cases.ground, cases.raman_lab, cases.dense_ops, cases.dense_kin])
def test_four_stages(gpu, make, size, precision):
    nx, ny = size
    print(f"[mixed tiles] four stages {make.__name__} {nx}x{ny} {precision}", flush=True)
    _check(gpu, _runs([functools.partial(make)], size), nx, ny, 1, precision)
