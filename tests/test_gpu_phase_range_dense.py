"""Dense potentials and coupling arrays on 256-point rows in every layout (GPU):
points one by one (complex128 radix 8 and 16), in blocks and in the split
layout, with the largest phase of the step at 0.9, 1.3 and (real time) 20
times the bound up to which the polynomials go without a range reduction. One full step against the oracle to the parity tests' tolerances
(complex128 1e-11, complex64 2e-4)."""

import numpy as np
import pytest

from cases import dense_ops
from oracle.reference_path import OraclePropagator
from spinor_gpe.pspinor.tensor_propagator import TensorPropagator

pytestmark = pytest.mark.gpu

BOUND = {'real': 0.785, 'imag': 0.346}
GAMMA = 1 / (2 + 2 ** (1 / 3))


@pytest.mark.parametrize('precision', ['c128', 'c64'])
@pytest.mark.parametrize('shape', [(2, 1), (4, 2), (8, 2), (16, 4), (4, -1)])
@pytest.mark.parametrize('time,peak', [('real', 0.9), ('real', 1.3), ('real', 20.0), ('imag', 0.9), ('imag', 1.3)])
def test_dense_phase_range(gpu, time, peak, shape, precision):
    ps, _, _ = dense_ops(mesh=(256, 256), r=(16, 16))
    n = [np.abs(p) ** 2 for p in ps.psi]
    top = max(float(np.max(ps.g_sc['uu'] * n[0] + ps.g_sc['ud'] * n[1])) / 2,
              float(np.max(ps.g_sc['dd'] * n[1] + ps.g_sc['ud'] * n[0])) / 2,
              max(float(np.max(np.abs(v))) for v in ps.pot_eng_spin), float(np.max(ps.coupling)) / 4)
    dt = peak * BOUND[time] / (top * (1 - 2 * GAMMA))
    print(f"[phase-range] dense {time} peak={peak} {shape} {precision} dt={dt:.4g}", flush=True)
    oracle = OraclePropagator(ps, dt, time=time)
    oracle.run(1)
    prop = TensorPropagator(ps, dt, 1, device=gpu, time=time, precision=precision, progress=False)
    prop._plan.tune(row_e=shape[0], row_rows=shape[1])  # pylint: disable=protected-access
    prop.full_step()
    got = np.stack([p.cpu().numpy() for p in prop.psik])
    want = np.stack(oracle.psik_numpy())
    err = float(np.linalg.norm(got - want) / np.linalg.norm(want))
    assert err < (1e-11 if precision == 'c128' else 2e-4), err
