"""fft_2d from several threads at once on lengths none of them has used before
(GPU): the context's factorizations and twiddle tables are made on first use
and shared by all threads. Against NumPy (1e-14 relative L2, as the transform
tests)."""

from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest
import torch

from spinor_gpe.pspinor import tensor_tools as ttools

pytestmark = pytest.mark.gpu

LENGTHS = [70, 84, 112, 132, 140, 154, 156, 168, 176, 182, 196, 198, 220, 224, 234, 252]


def test_first_use_in_threads(gpu):
    rng = np.random.default_rng(0)
    host = [[rng.normal(size=(n, 2 * n)) + 1j * rng.normal(size=(n, 2 * n)) for _ in range(2)] for n in LENGTHS]
    dev = [[torch.as_tensor(p, device=gpu) for p in pair] for pair in host]
    torch.cuda.synchronize()

    def call(i):
        return ttools.fft_2d(dev[i % len(dev)], (0.1, 0.2))

    with ThreadPoolExecutor(8) as pool:
        got = list(pool.map(call, range(4 * len(dev))))
    torch.cuda.synchronize()
    for i, out in enumerate(got):
        want = ttools.fft_2d(host[i % len(host)], (0.1, 0.2))
        for g, w in zip(out, want):
            assert np.linalg.norm(g.cpu().numpy() - w) < 1e-14 * np.linalg.norm(w), LENGTHS[i % len(host)]
