"""norm() of tensors (GPU): the out-of-place path against the in-place C entry
(same kernels, so bit for bit), with the inputs left untouched; grids below and
above the reduction's 1024 blocks, odd sizes; slices, offset rows and tensors
that require a gradient against NumPy (a few roundings per element: 4e-15
complex128, 4e-6 complex64). Two streams at once, each with its own scratch."""

import ctypes

import numpy as np
import pytest
import torch

from spinor_gpe import _native as nat
from spinor_gpe.pspinor import tensor_tools as ttools

pytestmark = pytest.mark.gpu


def _pair(shape, dtype, gpu, seed=0):
    rng = np.random.default_rng(seed)
    return [torch.as_tensor(rng.normal(size=shape) + 1j * rng.normal(size=shape), dtype=dtype, device=gpu)
            for _ in range(2)]


@pytest.mark.parametrize('dtype', [torch.complex128, torch.complex64])
@pytest.mark.parametrize('shape', [(1, 1), (3, 5), (64, 96), (511, 513), (700, 900)])
def test_same_as_in_place(gpu, shape, dtype):
    psi = _pair(shape, dtype, gpu)
    keep = [p.clone() for p in psi]
    got, dens = ttools.norm(psi, 0.05, 1234.5)
    prec = nat.precision_of(dtype)
    ref = [p.clone() for p in psi]
    dref = [torch.empty(shape, dtype=nat.REAL_DTYPE[prec], device=gpu) for _ in range(2)]
    ptr = [ctypes.c_void_p(t.data_ptr()) for t in ref + dref]
    nat.check(nat.lib().sgpe_norm(nat.Context.get(gpu).handle, prec, *shape, ptr[0], ptr[1], 0.05, 1234.5, ptr[2],
                                  ptr[3], None))
    torch.cuda.synchronize()
    for a, b in zip(got + dens + psi, ref + dref + keep):
        assert torch.equal(a, b)


@pytest.mark.parametrize('dtype', [torch.complex128, torch.complex64])
@pytest.mark.parametrize('kind', ['grad', 'sliced', 'offset'])
def test_other_pairs(gpu, kind, dtype):
    """Pairs that require a gradient or are slices of wider arrays are copied
    first; contiguous rows at an odd offset of a larger array are not."""
    psi = _pair((49, 161), dtype, gpu)
    if kind == 'grad':
        psi = [p.requires_grad_() for p in psi]
    elif kind == 'sliced':
        psi = [p[:, 1::2] for p in psi]
    else:
        psi = [p[1:] for p in psi]
    assert all(p.is_contiguous() for p in psi) == (kind != 'sliced')
    host = [p.detach().cpu().numpy().astype(np.complex128) for p in psi]
    got, dens = ttools.norm(psi, 0.05, 12.5)
    want, dwant = ttools.norm(host, 0.05, 12.5)
    tol = 4e-15 if dtype == torch.complex128 else 4e-6
    for g, w in zip(got + dens, want + dwant):
        assert np.linalg.norm(g.detach().cpu().numpy() - w) <= tol * np.linalg.norm(w)
    for p, h in zip(psi, host):
        assert np.array_equal(p.detach().cpu().numpy(), h)


def test_two_streams(gpu):
    pairs = [_pair((600, 640), torch.complex128, gpu, seed=s) for s in (1, 2)]
    want = [ttools.norm([p.cpu().numpy() for p in pair], 0.1, 50.0)[0] for pair in pairs]
    streams = [torch.cuda.Stream() for _ in pairs]
    torch.cuda.synchronize()
    outs = [[], []]
    for _ in range(10):
        for k, (st, pair) in enumerate(zip(streams, pairs)):
            with torch.cuda.stream(st):
                outs[k].append(ttools.norm(pair, 0.1, 50.0)[0])
    torch.cuda.synchronize()
    for k in range(2):
        for got in outs[k]:
            for g, w in zip(got, want[k]):
                assert np.linalg.norm(g.cpu().numpy() - w) <= 4e-15 * np.linalg.norm(w)
