"""Kinetic factors of the column pass (GPU): every pair of neighbouring
sub-steps (outer and inner in every order), the pass that starts from k-space,
the closing pass, and the sum for the populations with and without a k-space
read-back between the steps; real and imaginary time, tables and dense kinetic
arrays, compiled and runtime-length columns. Against the oracle to the parity
tests' tolerances (state 1e-11 / 2e-4, populations 1e-11 / 1e-5 of the atoms)."""

import functools

import numpy as np
import pytest
import torch

from oracle.reference_path import OraclePropagator, calc_pops
from spinor_gpe.engine.plan import InstanceSpec, Plan

from cases import dense_kin, dense_ops, ground, raman_lab, raman_rot

pytestmark = pytest.mark.gpu

MAKERS = {'ground': ground, 'lab': raman_lab, 'rot': raman_rot, 'dense_ops': dense_ops, 'dense_kin': dense_kin,
          'ground_96x160': functools.partial(ground, mesh=(96, 160)),
          'lab_80x96': functools.partial(raman_lab, mesh=(80, 96)),
          'dense_kin_96': functools.partial(dense_kin, mesh=(96, 96))}


@pytest.mark.parametrize('precision', ['c128', 'c64'])
@pytest.mark.parametrize('flip', [False, True])
@pytest.mark.parametrize('name', sorted(MAKERS))
def test_pairs(gpu, name, flip, precision):
    """flip: the other time mode on the same operators."""
    ps, time, dt = MAKERS[name]()
    if flip:
        time = 'real' if time == 'imag' else 'imag'
    print(f"[kinetic-pairs] {name} {time} {precision}", flush=True)
    oracle = OraclePropagator(ps, dt, time=time)
    spec = InstanceSpec.from_spin(ps, time, dt)
    plan = Plan(gpu, precision, spec.ny, spec.nx, 1)
    state = plan.new_state(ps.psik)
    plan.set_slot(0, spec, state)
    tol = 1e-11 if precision == 'c128' else 2e-4

    def check():
        plan.sync()
        want = np.stack(oracle.psik_numpy())
        err = float(np.linalg.norm(state.cpu().numpy() - want) / np.linalg.norm(want))
        assert err < tol, err

    subs = {0: (oracle.dt_out, oracle.eng_out), 1: (oracle.dt_in, oracle.eng_in)}
    for which in (1, 1, 0, 0, 1):
        plan.single_step(which)
        oracle.single_step(*subs[which])
    check()
    pops = torch.zeros((4, 2), dtype=torch.float64, device=gpu)
    plan.set_run(0, pops)
    ref = []
    for n in (1, 3):
        plan.full_steps(n)
        for _ in range(n):
            oracle.full_step()
            ref.append([float(p) for p in calc_pops(oracle.psik, oracle.space['dv_k'])])
        check()
    perr = float(np.max(np.abs(pops.cpu().numpy() - np.array(ref))) / ps.atom_num)
    assert perr < (1e-11 if precision == 'c128' else 1e-5), perr
