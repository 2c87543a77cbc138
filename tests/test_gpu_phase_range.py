"""Interaction phases across the bound up to which the row pass takes its
sin/cos and exp polynomials without a range reduction (GPU): every wave below
the bound, some waves on either side of it, most above it; real and imaginary
time, with and without a coupling phase, separable and dense operators, rows
taken point by point (complex128 radix 8) and in blocks. One full step against
the oracle to the parity tests' tolerances (complex128 1e-11, complex64 2e-4);
the state is normalized every sub-step, so its size does not scale them."""

import numpy as np
import pytest

from oracle.reference_path import OraclePropagator
from spinor_gpe.pspinor.tensor_propagator import TensorPropagator

from cases import dense_ops, ground, raman_lab, raman_rot

pytestmark = pytest.mark.gpu

BOUND = {'real': 0.785, 'imag': 0.346}
GAMMA = 1 / (2 + 2 ** (1 / 3))


@pytest.mark.parametrize('precision', ['c128', 'c64'])
@pytest.mark.parametrize('peak', [0.9, 1.3, 20.0])
@pytest.mark.parametrize('shape', [None, (8, 2), (4, 1)])
@pytest.mark.parametrize('make', [ground, raman_lab, raman_rot, dense_ops])
@pytest.mark.parametrize('time', ['real', 'imag'])
def test_phase_range(gpu, time, make, shape, peak, precision):
    mesh = (128, 128) if make is dense_ops else (256, 256)
    if shape is not None and mesh != (256, 256):
        pytest.skip('row shapes listed for 256 points')
    ps, _, _ = make(mesh=mesh) if make is not dense_ops else make()
    n = [np.abs(p) ** 2 for p in ps.psi]
    top = max(float(np.max(ps.g_sc['uu'] * n[0] + ps.g_sc['ud'] * n[1])),
              float(np.max(ps.g_sc['dd'] * n[1] + ps.g_sc['ud'] * n[0])))
    dt = peak * BOUND[time] / (top * (1 - 2 * GAMMA) / 2)
    if time == 'imag' and make is not ground:
        dt = min(dt, 1.2 * BOUND[time] / (top * (1 - 2 * GAMMA) / 2))  # the coupling's growth stays representable
    print(f"[phase-range] {make.__name__} {time} peak={peak} {shape} {precision} dt={dt:.4g}", flush=True)
    oracle = OraclePropagator(ps, dt, time=time)
    oracle.run(1)
    prop = TensorPropagator(ps, dt, 1, device=gpu, time=time, precision=precision, progress=False)
    if shape is not None:
        prop._plan.tune(row_e=shape[0], row_rows=shape[1])  # pylint: disable=protected-access
    prop.full_step()
    got = np.stack([p.cpu().numpy() for p in prop.psik])
    want = np.stack(oracle.psik_numpy())
    err = float(np.linalg.norm(got - want) / np.linalg.norm(want))
    assert err < (1e-11 if precision == 'c128' else 2e-4), err
