"""Kernels that multiply float32 values as three bf16 limbs, against 64 bits, through the C ABI."""

from __future__ import annotations

import ctypes

import pytest
import torch

from flux_amd import _native

pytestmark = pytest.mark.gpu


def _randn(*shape, seed, std=1.0):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * std).float()


def _linear(a, w, residual, device):
    m, k = a.shape
    n = w.shape[0]
    a, w = a.to(device), w.to(device)
    r = None if residual is None else residual.to(device)
    c = torch.empty(m, n, device=device)
    _native.check(_native.load().flux_linear_f32(a.data_ptr(), w.data_ptr(), _native.ptr(r), c.data_ptr(), m, n, k,
                                                 _native.current_stream(device)))
    torch.cuda.synchronize()
    return c.cpu()


@pytest.mark.parametrize("m,n,k", [
    (1, 64, 16), (65, 192, 48),          # one stage; an odd number of stages, a half-empty column tile
    (1793, 576, 576), (2049, 576, 1536),  # 64-row tiles, the last of one row
    (1025, 3072, 64), (3073, 960, 576),   # 128-row tiles
    (8193, 3072, 32),                     # 256-row tiles
])
def test_limb_linear_error_bound(gpu_device, m, n, k):
    a, w, r = _randn(m, k, seed=1), _randn(n, k, seed=2, std=0.05), _randn(m, n, seed=3)
    exact = a.double() @ w.double().T
    size = a.double().abs() @ w.double().abs().T
    # Each limb product is exact.  The leading limbs' accumulator is rounded once per 16 K values
    # at no more than the size of the sum of magnitudes, the small products' five times as often
    # at 2^-8 of it; the dropped products are below 2^-25 of it.  Two units in the last place per
    # rounding leave room for an instruction that truncates what it adds up.
    bound = size * (k / 16 * (1 + 5 / 256) + 2) * 2.0 ** -22
    for residual in (None, r):
        c = _linear(a, w, residual, gpu_device).double()
        want = exact if residual is None else exact + r.double()
        limit = bound if residual is None else bound + want.abs() * 2.0 ** -23
        assert torch.all((c - want).abs() <= limit)


def test_limb_linear_keeps_float32_range(gpu_device):
    # What bf16 limbs cannot carry: infinities, values above the largest bf16, and rows of
    # denormals.  Every other row of the tile is what it is without them.
    m, n, k = 2048, 576, 576
    a, w = _randn(m, k, seed=4), _randn(n, k, seed=5, std=0.05)
    a[3, 7] = float("inf")
    a[4, 9] = float("-inf")
    a[5, 11] = float("nan")
    a[6] = 0.0
    a[6, 2] = 3.4e38
    a[700] = 1e-41
    c = _linear(a, w, None, gpu_device)
    assert torch.equal(c[3], torch.sign(w[:, 7]) * float("inf"))
    assert torch.equal(c[4], -torch.sign(w[:, 9]) * float("inf"))
    assert torch.all(torch.isnan(c[5]))
    torch.testing.assert_close(c[6].double(), 3.4e38 * w[:, 2].double(), rtol=1e-6, atol=0)
    torch.testing.assert_close(c[700].double(), a[700].double() @ w.double().T, rtol=0, atol=1e-42 * k)
    rows = [r for r in range(m) if r not in (3, 4, 5, 6, 700)]
    torch.testing.assert_close(c[rows].double(), a[rows].double() @ w.double().T, rtol=1e-4, atol=1e-4)
