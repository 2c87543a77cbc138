"""Mixed-radix kernels (GPU): lengths that use every radix from 2 to 16, two to
five stages, the shortest and longest, lengths that just miss them (a prime
factor above 13, fewer than 32 points) and stay with the runtime-length
kernels, and tiles of odd width. Transforms against NumPy (relative L2: rounding
of log2 N levels, 1e-14 complex128 and 5e-6 complex64 with a margin of ten);
one full step in imaginary and two sub-steps in real time against the oracle to
the parity tests' tolerances."""

import functools

import numpy as np
import pytest
import torch

from oracle.reference_path import OraclePropagator
from spinor_gpe.engine.plan import InstanceSpec, Plan
from spinor_gpe.pspinor import tensor_tools as ttools

from cases import dense_ops, ground, raman_lab, raman_rot

pytestmark = pytest.mark.gpu

SIZES = [(32, 48), (34, 36), (30, 32), (66, 78), (98, 90), (104, 110), (126, 182), (154, 130), (210, 242), (286, 338),
         (225 * 2, 360), (486, 500), (750, 1458), (1250, 98), (1386, 66), (1694, 42), (2000, 54), (2028, 50), (2048, 6),
         (62, 2028), (70, 1950), (38, 2000), (6, 1250), (1000, 1000)]


@pytest.mark.parametrize('precision', ['c128', 'c64'])
@pytest.mark.parametrize('size', SIZES, ids=str)
def test_transforms(gpu, size, precision):
    ny, nx = size
    print(f"[mixed-radix] fft {ny}x{nx} {precision}", flush=True)
    rng = np.random.default_rng(ny * 4096 + nx)
    dtype = torch.complex128 if precision == 'c128' else torch.complex64
    psi = [torch.as_tensor(rng.normal(size=size) + 1j * rng.normal(size=size), dtype=dtype, device=gpu)
           for _ in range(2)]
    host = [p.cpu().numpy().astype(np.complex128) for p in psi]
    dr = (0.3, 0.2)
    tol = 1e-14 if precision == 'c128' else 5e-6
    for got, want in ((ttools.fft_2d(psi, dr), ttools.fft_2d(host, dr)),
                      (ttools.ifft_2d(psi, dr), ttools.ifft_2d(host, dr))):
        for g, w in zip(got, want):
            err = float(np.linalg.norm(g.cpu().numpy() - w) / np.linalg.norm(w))
            assert err < tol, err


@pytest.mark.parametrize('precision', ['c128', 'c64'])
@pytest.mark.parametrize('slots', [1, 3])
@pytest.mark.parametrize('size', [(32, 34), (90, 98), (126, 110), (64, 150), (154, 128), (286, 182), (104, 338)], ids=str)
@pytest.mark.parametrize('make', [ground, raman_rot, raman_lab, dense_ops])
def test_step(gpu, make, size, slots, precision):
    ny, nx = size
    print(f"[mixed-radix] step {make.__name__} {ny}x{nx} x{slots} {precision}", flush=True)
    ps, time, dt = functools.partial(make, mesh=(nx, ny))()
    oracle = OraclePropagator(ps, dt, time=time)
    oracle.full_step()
    oracle.single_step(oracle.dt_in, oracle.eng_in)
    spec = InstanceSpec.from_spin(ps, time, dt)
    plan = Plan(gpu, precision, ny, nx, slots)
    states = [plan.new_state(ps.psik) for _ in range(slots)]
    for i, s in enumerate(states):
        plan.set_slot(i, spec, s)
    plan.full_steps(1)
    plan.single_step(1)
    plan.sync()
    want = np.stack(oracle.psik_numpy())
    for s in states:
        err = float(np.linalg.norm(s.cpu().numpy() - want) / np.linalg.norm(want))
        assert err < (1e-11 if precision == 'c128' else 2e-4), err
