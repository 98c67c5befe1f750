"""Kernels that multiply float32 values as three bf16 limbs, against 64 bits, through the C ABI."""

from __future__ import annotations

import ctypes
import math

import pytest
import torch

from flux_amd import _native

pytestmark = pytest.mark.gpu


def _randn(*shape, seed, std=1.0):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * std).float()


def _rel(got, want):
    return float((got - want).norm() / want.norm())


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
    (1025, 3072, 64), (3073, 960, 576), (8193, 3072, 32),  # 128-row tiles
    (7937, 3072, 32), (2501, 3072, 576),  # 256-row tiles, the last of one row and of 197
])
def test_limb_linear_error_bound(gpu_device, m, n, k):
    a, w, r = _randn(m, k, seed=1), _randn(n, k, seed=2, std=0.05), _randn(m, n, seed=3)
    exact = a.double() @ w.double().T
    size = a.double().abs() @ w.double().abs().T
    # Each limb product is exact.  The leading limbs' accumulator is rounded once per 16 K values
    # at no more than the size of the sum of magnitudes, the small products' five times as often
    # at 2^-8 of it; the dropped products are below 2^-23 of it (a second times a third limb, twice,
    # of at most 2^-8 and 2^-16 of their values).  Two units in the last place per rounding leave
    # room for an instruction that truncates what it adds up.
    bound = size * (k / 16 * (1 + 5 / 256) + 2) * 2.0 ** -22
    # In the norm: a rounding error is 2^-24 / sqrt(3) of what is rounded, and the partial sums of
    # random products grow as the root of their number, so K / 16 of them add up to
    # sqrt(K / 32) of that; half as much again, and one for the last rounding.  Without the third
    # limb the error is about ten times this bound.
    norm = (1.5 * math.sqrt(k / 32) + 1) * 2.0 ** -24 / math.sqrt(3)
    for residual in (None, r):
        c = _linear(a, w, residual, gpu_device).double()
        want = exact if residual is None else exact + r.double()
        limit = bound if residual is None else bound + want.abs() * 2.0 ** -23
        assert torch.all((c - want).abs() <= limit)
        if residual is None and k >= 576:
            assert _rel(c, want) < norm


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
    # Float32 rounds K / 2 sums of two products to multiples of 2^-149, by at most half of one, and
    # the result and the products once more; the outputs are thousands of them.
    want = a[700].double() @ w.double().T
    torch.testing.assert_close(c[700].double(), want, rtol=0, atol=k * 2.0 ** -149)
    assert torch.all(c[700][want.abs() > k * 2.0 ** -149] != 0.0) and float(want.abs().max()) > 10 * k * 2.0 ** -149
    rows = [r for r in range(m) if r not in (3, 4, 5, 6, 700)]
    torch.testing.assert_close(c[rows].double(), a[rows].double() @ w.double().T, rtol=1e-4, atol=1e-4)


def _rows_call(name, x, w, device):
    """The GEMM `name` on rows `x`, and the same with float64 products."""
    rows = x.shape[0]
    if name == "linear":
        return _linear(x, w, None, device), x.double() @ w.double().T
    lib, stream = _native.load(), _native.current_stream(device)
    exact = x.double() @ w.double().T
    x, w = x.to(device), w.to(device)
    if name == "gate_up":
        out = torch.empty(rows, 1536, device=device)
        _native.check(lib.flux_gate_up_swiglu_rows_f32(x.data_ptr(), w.data_ptr(), out.data_ptr(), rows, stream))
        gate, up = exact.chunk(2, dim=-1)
        want = gate / (1 + torch.exp(-gate)) * up
    else:
        # cos = 1, sin = 0: the rotation adds 0 times the paired column.
        cos, sin = torch.ones(rows, 64, device=device), torch.zeros(rows, 64, device=device)
        out = torch.empty(15, rows, 64, device=device)
        _native.check(lib.flux_qkv_rope_cache_rows_f32(x.data_ptr(), w.data_ptr(), cos.data_ptr(), sin.data_ptr(),
                                                       rows, out[:9].data_ptr(), out[9:12].data_ptr(),
                                                       out[12:].data_ptr(), rows, stream))
        heads = exact.view(rows, 15, 64).transpose(0, 1)
        paired = torch.cat((-heads[:12, :, 32:], heads[:12, :, :32]), dim=-1)
        want = torch.cat((heads[:12] + paired.float() * 0.0, heads[12:]))
    torch.cuda.synchronize()
    return out.cpu(), want


@pytest.mark.parametrize("name,n", [("linear", 576), ("gate_up", 3072), ("qkv", 960)])
def test_limb_gemm_infinity_and_nan(gpu_device, name, n):
    # An infinity in one row and a NaN in another, in different tiles; all others as without.
    x, w = _randn(2500, 576, seed=34), _randn(n, 576, seed=35, std=0.05)
    x[3, 7], x[2499, 11] = float("inf"), float("nan")
    got, want = _rows_call(name, x, w, gpu_device)
    want = want.float()
    odd = ~torch.isfinite(want)
    assert int(odd.sum()) == 2 * (want.shape[-1] if name != "qkv" else 960)
    torch.testing.assert_close(got[odd], want[odd], rtol=0, atol=0, equal_nan=True)
    torch.testing.assert_close(got[~odd], want[~odd], rtol=5e-4, atol=1e-4)


# 2500 rows: the limb kernel under each epilogue.
@pytest.mark.parametrize("name,n", [("linear", 576), ("gate_up", 3072), ("qkv", 960)])
def test_limb_gemm_overflow_is_infinite(gpu_device, name, n):
    # Products of finite values that overflow: the leading limbs' to one infinity, of a small pair
    # of limbs possibly to the other.
    x, w = _randn(2500, 576, seed=30), _randn(n, 576, seed=31, std=0.05)
    if name == "gate_up":
        w[:1536, [7, 11]] = 0.0  # the gates stay ordinary
    up = n - 100  # a column of up, of a value head, or any
    x[3, 7], w[up, 7] = 1.3e25, 1.7e25
    x[2499, 11], w[up + 1, 11] = 1.234e22, -5.678e22
    got, want = _rows_call(name, x, w, gpu_device)
    want = want.float()
    assert int(torch.isinf(want).sum()) == 2
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(got[torch.isinf(want)], want[torch.isinf(want)])
    ordinary = [r for r in range(2500) if r not in (3, 2499)]
    got, want = ((t.movedim(-2, 0)[ordinary]).flatten(1) for t in (got, want))
    columns = [c for c in range(want.shape[1]) if c not in (up % want.shape[1], up % want.shape[1] + 1)]
    torch.testing.assert_close(got[:, columns], want[:, columns], rtol=5e-4, atol=1e-4)


@pytest.mark.parametrize("small", [2.0 ** -120, 1e-38, 1e-41])
@pytest.mark.parametrize("of", ["x", "w"])
@pytest.mark.parametrize("name,n", [("linear", 576), ("gate_up", 3072), ("qkv", 960)])
def test_limb_gemm_small_magnitudes(gpu_device, name, n, of, small):
    # Rows, or weights, of which bf16 limbs keep only the leading bits or none: as close as others
    # (the float32 instruction is at 4.4e-7 for K = 576; SwiGLU multiplies two such sums).
    x, w = _randn(2500, 576, seed=32), _randn(n, 576, seed=33, std=0.05)
    if of == "x":
        x[1200:1300] *= small
        w *= 2.0 ** 100
    else:
        w *= small
        x *= 2.0 ** 100
    got, want = _rows_call(name, x, w, gpu_device)
    if of == "x":
        rows = (lambda t: t[:, 1200:1300]) if name == "qkv" else (lambda t: t[1200:1300])
        got, want = rows(got), rows(want)
    assert _rel(got.double(), want) < 1e-6


def _attention(q, k, v, device):
    lib = _native.load()
    seq = q.shape[1]
    need = ctypes.c_int64()
    _native.check(lib.flux_prefill_attention_workspace_bytes(seq, ctypes.byref(need)))
    q, k, v = q.to(device), k.to(device), v.to(device)
    workspace = torch.empty(max(1, need.value // 4), device=device)
    out = torch.empty(seq, 576, device=device)
    _native.check(lib.flux_prefill_attention_f32(q.data_ptr(), k.data_ptr(), v.data_ptr(), seq, k.shape[1], 0.125,
                                                 workspace.data_ptr(), out.data_ptr(),
                                                 _native.current_stream(device)))
    torch.cuda.synchronize()
    return out.cpu().view(seq, 9, 64).transpose(0, 1).double()


def _attention64(q, k, v):
    seq = q.shape[1]
    k, v = (t.double()[:, :seq].repeat_interleave(3, 0) for t in (k, v))
    scores = q.double() @ k.transpose(1, 2) * 0.125
    scores.masked_fill_(torch.ones(seq, seq, dtype=torch.bool).triu(1), float("-inf"))
    return torch.softmax(scores, -1) @ v


# 896 | 897: below and above the shortest limb prompt; 961: a last key tile of one row; 1153: a
# last query tile of one row; 2400: chunks of 8 tiles, the last one partial.
@pytest.mark.parametrize("seq", [896, 897, 961, 1153, 2400])
def test_limb_attention_is_as_exact_as_float32(gpu_device, seq):
    q, k, v = (_randn(h, seq + 7 * (h == 3), 64, seed=10 + i) for i, h in enumerate((9, 3, 3)))
    want = _attention64(q, k, v)
    got = _attention(q, k, v, gpu_device)
    # Scores of 64 products and at most seq weights that sum to one: a relative 1e-6 is two units
    # in the last place of float32 for every ninth of them.
    assert float((got - want).norm() / want.norm()) < 1e-6
    torch.testing.assert_close(got, want, rtol=2e-4, atol=2e-5)


def test_limb_attention_keeps_float32_range(gpu_device):
    # A key that no query can see (its score is -inf), one above the largest bf16 and a value that
    # is infinite: the blocks that read them take the float32 instruction, the others do not.
    seq = 1500
    q, k, v = _randn(9, seq, 64, seed=20), _randn(3, seq, 64, seed=21), _randn(3, seq, 64, seed=22)
    q[:, :, 0] = -q[:, :, 0].abs() - 0.1
    k[0, 700, 0] = float("inf")
    k[1, 3, 0] = 3.4e38
    v[2, 1000, 5] = float("inf")
    got = _attention(q, k, v, gpu_device)
    seen = k.clone()
    seen[0, 700] = 0.0
    want = _attention64(q, k, v)
    k0 = seen[0].double()
    scores = q[:3].double() @ k0.T * 0.125
    scores[:, :, 700] = float("-inf")
    scores.masked_fill_(torch.ones(seq, seq, dtype=torch.bool).triu(1), float("-inf"))
    want[:3] = torch.softmax(scores, -1) @ v[0].double()
    torch.testing.assert_close(got[:6], want[:6], rtol=2e-4, atol=2e-5)
    assert torch.all(got[6:, 1000:, 5] == float("inf"))
    rest = [d for d in range(64) if d != 5]
    torch.testing.assert_close(got[6:, :, rest], want[6:, :, rest], rtol=2e-4, atol=2e-5)


def test_limb_attention_nan(gpu_device):
    # A NaN key or value reaches every query that sees its row, a NaN query its own row only.
    seq = 1500
    q, k, v = _randn(9, seq, 64, seed=37), _randn(3, seq, 64, seed=38), _randn(3, seq, 64, seed=39)
    want = _attention64(q, k, v)
    k[0, 1200, 3] = float("nan")
    v[1, 1300, 4] = float("nan")
    q[8, 70, 5] = float("nan")
    got = _attention(q, k, v, gpu_device)
    assert torch.all(torch.isnan(got[:3, 1200:])) and torch.all(torch.isnan(got[3:6, 1300:, 4]))
    assert torch.all(torch.isnan(got[8, 70]))
    seen = torch.ones(9, seq, 64, dtype=torch.bool)
    seen[:3, 1200:] = False
    # Masked weights are exactly zero, and zero times NaN is NaN: the value's 64-key tile too.
    seen[3:6, 1280:, 4] = False
    seen[8, 70] = False
    torch.testing.assert_close(got[seen], want[seen], rtol=2e-4, atol=2e-5)


def test_limb_attention_overflow_is_infinite(gpu_device):
    # Scores whose products overflow to minus infinity, a small pair of limbs' to plus infinity:
    # queries from 1000 on cannot see key 700.
    seq = 1500
    q, k, v = _randn(9, seq, 64, seed=40), _randn(3, seq, 64, seed=41), _randn(3, seq, 64, seed=42)
    q[:3, :, 0], k[0, :, 0] = 0.0, 0.0
    q[:3, 1000:, 0], k[0, 700, 0] = 1.3e25, -1.7e25
    got = _attention(q, k, v, gpu_device)
    want = _attention64(q, k, v)  # a score of -4e49 has no weight in float64 either
    torch.testing.assert_close(got, want, rtol=2e-4, atol=2e-5)


def test_limb_attention_small_magnitudes(gpu_device):
    # Keys, queries and values of which bf16 limbs keep only the leading bits, one per KV head; every
    # output is as close as with ordinary magnitudes.
    seq = 1100
    q, k, v = _randn(9, seq, 64, seed=43), _randn(3, seq, 64, seed=44), _randn(3, seq, 64, seed=45)
    k[0] *= 2.0 ** -120
    q[:3] *= 2.0 ** 120
    k[1] *= 2.0 ** 122
    q[3:6] *= 2.0 ** -122
    v[2] *= 2.0 ** -121
    got, want = _attention(q, k, v, gpu_device), _attention64(q, k, v)
    for g in range(3):
        assert _rel(got[3 * g:3 * g + 3], want[3 * g:3 * g + 3]) < 1e-6


def test_limb_attention_small_weights(gpu_device):
    # Every query's weight is on the first key, whose values are zero; the outputs are the others',
    # with weights of about 2^-123.  A score of -123 is known to half a unit in the last place,
    # 2^-18, and so are these weights to 2.6e-6.
    seq = 1100
    q, k, v = _randn(9, seq, 64, seed=46, std=0.1), _randn(3, seq, 64, seed=47), _randn(3, seq, 64, seed=48)
    q[:, :, 0], k[:, :, 0] = 10.0, 0.0
    k[:, 0] = 0.0
    k[:, 0, 0] = 123 * math.log(2) / 1.25
    v[:, 0] = 0.0
    got, want = _attention(q, k, v, gpu_device), _attention64(q, k, v)
    assert _rel(got[:, 64:], want[:, 64:]) < 1e-5
