"""Split steps on the runtime-length kernels of both axes (GPU): lengths with a
prime factor above 13 or below 32 points, which no other kernel takes (34 = 2 *
17, 38 = 2 * 19, 62 = 2 * 31, 46 = 2 * 23, 22 and 26). Every pair of neighbouring
sub-steps, the pass that starts from k-space, the closing pass and the
populations with and without a read-back between the steps; real and imaginary
time; tables, dense kinetic, potential and coupling arrays; a sweep with its
energies; phases of up to 2e6 rad. Against the oracle to the parity tests'
tolerances (state 1e-11 / 2e-4, populations 1e-11 / 1e-5 of the atoms)."""

import functools

import numpy as np
import pytest
import torch

import cases
from oracle import energy as oe
from oracle.reference_path import OraclePropagator, calc_pops
from spinor_gpe.engine.plan import InstanceSpec, Plan
from spinor_gpe.engine.sweep import Sweep

pytestmark = pytest.mark.gpu

MAKERS = {'ground': functools.partial(cases.ground, mesh=(34, 38)),
          'lab': functools.partial(cases.raman_lab, mesh=(62, 46)),
          'rot': functools.partial(cases.raman_rot, mesh=(22, 26)),
          'dense_ops': functools.partial(cases.dense_ops, mesh=(62, 46)),
          'dense_kin': functools.partial(cases.dense_kin, mesh=(38, 34))}


def _rel(got, want):
    return float(np.linalg.norm(got - want) / np.linalg.norm(want))


@pytest.mark.parametrize('precision', ['c128', 'c64'])
@pytest.mark.parametrize('slots', [1, 2])
@pytest.mark.parametrize('flip', [False, True])
@pytest.mark.parametrize('name', sorted(MAKERS))
def test_sub_steps(gpu, name, flip, slots, precision):
    """flip: the other time mode on the same operators."""
    ps, time, dt = MAKERS[name]()
    if flip:
        time = 'real' if time == 'imag' else 'imag'
    print(f"[runtime-length] {name} {time} x{slots} {precision}", flush=True)
    oracle = OraclePropagator(ps, dt, time=time)
    spec = InstanceSpec.from_spin(ps, time, dt)
    plan = Plan(gpu, precision, spec.ny, spec.nx, slots)
    tuning = plan.tuning()
    assert tuning[0] == 0 and tuning[2] == 0
    states = [plan.new_state(ps.psik) for _ in range(slots)]
    for i, st in enumerate(states):
        plan.set_slot(i, spec, st)
    tol = 1e-11 if precision == 'c128' else 2e-4

    def check():
        plan.sync()
        want = np.stack(oracle.psik_numpy())
        for st in states:
            assert _rel(st.cpu().numpy(), want) < tol

    subs = {0: (oracle.dt_out, oracle.eng_out), 1: (oracle.dt_in, oracle.eng_in)}
    for which in (1, 1, 0, 0, 1):
        plan.single_step(which)
        oracle.single_step(*subs[which])
    check()
    pops = torch.zeros((slots, 4, 2), dtype=torch.float64, device=gpu)
    for i in range(slots):
        plan.set_run(i, pops[i])
    ref = []
    for n in (1, 3):
        plan.full_steps(n)
        for _ in range(n):
            oracle.full_step()
            ref.append([float(p) for p in calc_pops(oracle.psik, oracle.space['dv_k'])])
        check()
    perr = float(np.max(np.abs(pops.cpu().numpy() - np.array(ref))) / ps.atom_num)
    assert perr < (1e-11 if precision == 'c128' else 1e-5), perr


@pytest.mark.parametrize('precision', ['c128', 'c64'])
def test_sweep(gpu, precision):
    """One captured graph over three such grids, with on-device energy checks."""
    print(f"[runtime-length] sweep {precision}", flush=True)
    spins = [cases.raman_rot(name=f'rl{i}', mesh=mesh, seed=30 + i)[0]
             for i, mesh in enumerate([(34, 38), (46, 62), (22, 26), (34, 38)])]
    sw = Sweep(gpu, precision, conv_tol=0.0, check_every=10, max_steps=30)
    for ps in spins:
        sw.add_spin(ps, 0.02)
    res, _ = sw.run()
    for ps, r in zip(spins, res):
        oracle = OraclePropagator(ps, 0.02, time='imag')
        oracle.run(30)
        assert r.steps == 30
        assert _rel(r.psik, np.stack(oracle.psik_numpy())) < (1e-11 if precision == 'c128' else 2e-4)
        own = oe.gp_energy(r.psik, ps.space['dr'], ps.kin_eng_spin, ps.pot_eng_spin, ps.g_sc, ps.coupling, None)
        assert r.energy['E_tot'] == pytest.approx(own['E_tot'], rel=1e-12 if precision == 'c128' else 1e-5)


def test_large_phases(gpu):
    """Potential phases of up to 2e6 rad, formed per point (as the test of this
    name on compiled grids does)."""
    print("[runtime-length] large phases", flush=True)
    ps, _, _ = cases.ground(name='rlbig', mesh=(34, 62), r=(8, 8))
    x, y = ps.space['x_mesh'], ps.space['y_mesh']
    ps.pot_eng = ps.pot_eng + 1e9 * (0.5 + 0.5 * np.sin(0.7 * x * y + 0.3 * x))
    oracle = OraclePropagator(ps, 2e-3, time='real')
    ref = oracle.run(5)
    res, _ = ps.real(2e-3, 5, 'cuda', progress=False)
    assert _rel(np.stack(res.psik), np.stack(oracle.psik_numpy())) < 1e-11
    assert np.max(np.abs(res.pops['vals'] - ref)) < 1e-11 * ps.atom_num
