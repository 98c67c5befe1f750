"""Short-prompt GEMMs on 16-row tiles at the edges of their tilings, against 64 bits, through the C ABI."""

from __future__ import annotations

import pytest
import torch

from flux_amd import _native

pytestmark = pytest.mark.gpu


def _randn(*shape, seed, std=1.0):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * std).float()


def _call(name, *args):
    _native.check(getattr(_native.load(), name)(*(a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args),
                                                _native.current_stream()))
    torch.cuda.synchronize()


# Sums of K float32 products: K / 4 matrix instructions of four each and twelve partial sums, one
# rounding each, of at most the sum of magnitudes.
def _bound(a, w):
    return (a.double().abs() @ w.double().abs().T) * (w.shape[1] / 4 + 12) * 2.0 ** -24


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 112, 113])  # 112 | 113: 16-column tiles | split kernel
def test_down_projection_rows(gpu_device, rows):
    a, w, r = _randn(rows, 1536, seed=1), _randn(576, 1536, seed=2, std=0.02), _randn(rows, 576, seed=3)
    out = torch.empty(rows, 576, device=gpu_device)
    _call("flux_linear_f32", a.to(gpu_device), w.to(gpu_device), r.to(gpu_device), out, rows, 576, 1536)
    want = a.double() @ w.double().T + r.double()
    assert torch.all((out.cpu().double() - want).abs() <= _bound(a, w) + want.abs() * 2.0 ** -23)


@pytest.mark.parametrize("rows", [1, 16, 31, 32, 33, 80, 81])  # half groups up to 32 rows, whole up to 80
def test_gate_up_rows(gpu_device, rows):
    x, w = _randn(rows, 576, seed=4), _randn(3072, 576, seed=5, std=0.02)
    out = torch.empty(rows, 1536, device=gpu_device)
    _call("flux_gate_up_swiglu_rows_f32", x.to(gpu_device), w.to(gpu_device), out, rows)
    gate, up = (x.double() @ w.double().T).chunk(2, dim=-1)
    torch.testing.assert_close(out.cpu().double(), gate * torch.sigmoid(gate) * up, rtol=5e-4, atol=2e-5)


@pytest.mark.parametrize("rows", [1, 16, 128, 129, 272, 273])  # half groups up to 128 rows, whole up to 272
def test_qkv_rows(gpu_device, rows):
    x, w = _randn(rows, 576, seed=6), _randn(960, 576, seed=7, std=0.02)
    cos, sin = _randn(rows, 64, seed=8), _randn(rows, 64, seed=9)
    q, k, v = (torch.full((h, rows, 64), float("nan"), device=gpu_device) for h in (9, 3, 3))
    _call("flux_qkv_rope_cache_rows_f32", x.to(gpu_device), w.to(gpu_device), cos.to(gpu_device), sin.to(gpu_device),
          rows, q, k, v, rows)
    heads = (x.double() @ w.double().T).view(rows, 15, 64).transpose(0, 1)
    turned = torch.cat((-heads[..., 32:], heads[..., :32]), dim=-1)
    rotated = heads * cos.double() + turned * sin.double()
    for got, want in ((q, rotated[:9]), (k, rotated[9:12]), (v, heads[12:])):
        torch.testing.assert_close(got.cpu().double(), want, rtol=1e-4, atol=1e-5)


# Widths that are multiples of 128: 64 x 64 tiles while at most 256 of them, limb tiles beyond.
@pytest.mark.parametrize("rows,n,k", [(1, 128, 64), (8192, 128, 64), (8193, 128, 64), (65, 3072, 64), (321, 3072, 96)])
def test_linear_rows_of_wide_tiles(gpu_device, rows, n, k):
    a, w, r = _randn(rows, k, seed=10), _randn(n, k, seed=11), _randn(rows, n, seed=12)
    out = torch.empty(rows, n, device=gpu_device)
    _call("flux_linear_f32", a.to(gpu_device), w.to(gpu_device), r.to(gpu_device), out, rows, n, k)
    want = a.double() @ w.double().T + r.double()
    assert torch.all((out.cpu().double() - want).abs() <= _bound(a, w) + want.abs() * 2.0 ** -23)
