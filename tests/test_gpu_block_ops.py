"""Residual add + RMSNorm and SwiGLU kernels against the reference's op sequence
(layers.py:13-40) in torch, at the edges of their row splits and alignments."""

from __future__ import annotations

import pytest
import torch

from helios_amd import ops
from tests.gpu_cases import say

pytestmark = pytest.mark.gpu

ULP = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}  # spacing of a value in [1, 2)


def _rms(x, w, eps):
    f = x.float()
    return (f * torch.rsqrt(f.pow(2).mean(-1, keepdim=True) + eps) * w).to(x.dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,hidden", [(1, 8), (3, 20), (130, 2048), (129, 2056), (5, 2560), (2, 8192), (2, 8200),
                                         (7, 4099)])
def test_add_rms_norm(device, rows, hidden, dtype):
    say("add_rms_norm", rows, hidden, dtype)
    g = torch.Generator(device=device).manual_seed(rows * hidden)
    x = torch.randn(1, rows, hidden, generator=g, device=device).to(dtype)
    y = (3 * torch.randn(1, rows, hidden, generator=g, device=device)).to(dtype)
    w = 1 + 0.1 * torch.randn(hidden, generator=g, device=device)
    for other in (None, y):
        total, normed = ops.add_rms_norm(x, other, w, 1e-6)
        want = x if other is None else x + y
        assert torch.equal(total, want)
        ref = _rms(want, w, 1e-6).float()
        # The fp32 statistics differ in the order of their sums only: one rounding step at most.
        assert ((normed.float() - ref).abs() <= ULP[dtype] * ref.abs() + 1e-7).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,ffn", [(1, 8), (3, 5), (33, 2056), (2, 9728), (9, 1023)])
def test_swiglu(device, rows, ffn, dtype):
    say("swiglu", rows, ffn, dtype)
    g = torch.Generator(device=device).manual_seed(rows * ffn)
    x = (6 * torch.randn(rows, 2 * ffn, generator=g, device=device)).to(dtype)
    x[0, :5] = torch.tensor([0.0, -0.0, 300.0, -300.0, -90.0], device=device).to(dtype)
    gate, up = x.chunk(2, dim=-1)
    ref = (torch.nn.functional.silu(gate) * up).float()
    got = ops.swiglu(x).float()
    # silu in fp32 to a few fp32 ulps either way, then two roundings: silu may round one
    # step apart, which the product carries into at most two of its own. Below the
    # smallest normal the step is absolute.
    tiny = torch.finfo(dtype).tiny
    assert ((got - ref).abs() <= 2 * ULP[dtype] * ref.abs() + 8 * tiny).all()


def test_swiglu_limits(device):
    say("swiglu limits")
    inf, nan = float("inf"), float("nan")
    gate = torch.tensor([inf, -inf, nan, 1.0, 1.0, 1e38, -1e38, 0.0], device=device).to(torch.bfloat16)
    up = torch.tensor([2.0, 2.0, 1.0, inf, nan, 1.0, 1.0, inf], device=device).to(torch.bfloat16)
    ref = (torch.nn.functional.silu(gate) * up).float()
    got = ops.swiglu(torch.cat((gate, up)).unsqueeze(0))[0].float()
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    keep = ~torch.isnan(ref)
    assert torch.equal(got[keep], ref[keep])


def test_add_rms_norm_and_swiglu_refuse_what_they_cannot_read(device):
    x = torch.zeros(2, 16, dtype=torch.bfloat16, device=device)
    w = torch.ones(16, device=device)
    with pytest.raises(ValueError):
        ops.add_rms_norm(x[:, ::2], None, w[:8], 1e-6)
    with pytest.raises(ValueError):
        ops.add_rms_norm(x, x[:1], w, 1e-6)
    with pytest.raises(ValueError):
        ops.add_rms_norm(x.float(), None, w, 1e-6)
    with pytest.raises(ValueError):
        ops.swiglu(x[:, :15])


def _parts(x, w, norm, eps, residual, swiglu):
    """The separate steps, rounding where they round."""
    h = x if norm is None else _rms(x, norm, eps)
    y = (h.double() @ w.double().t()).to(x.dtype)
    if swiglu:
        gate, up = y.chunk(2, dim=-1)
        return torch.nn.functional.silu(gate) * up
    return y if residual is None else residual + y


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,cols,k", [(1, 16, 64), (8, 48, 192), (9, 2560, 2560), (16, 32, 704), (15, 16, 9728)])
def test_block_linear(device, rows, cols, k, dtype):
    """Row counts around the half tiles, K slices that are empty, uneven and long, beyond
    the part of a row that the norm's statistics hold in registers."""
    say("block_linear", rows, cols, k, dtype)
    g = torch.Generator(device=device).manual_seed(rows + cols + k)
    x = torch.randn(1, rows, k, generator=g, device=device).to(dtype)
    w = (torch.randn(2 * cols, k, generator=g, device=device) * k ** -0.5).to(dtype)
    norm = 1 + 0.1 * torch.randn(k, generator=g, device=device)
    residual = torch.randn(1, rows, cols, generator=g, device=device).to(dtype)
    for n in (None, norm):
        for kw in (dict(), dict(residual=residual), dict(swiglu=True)):
            wt = w if kw.get("swiglu") else w[:cols]
            got = ops.block_linear(x, wt, norm_weight=n, eps=1e-6, **kw).float()
            ref = _parts(x, wt, n, 1e-6, kw.get("residual"), kw.get("swiglu", False)).float()
            # fp32 sums of products of size 1/sqrt(k): y is right to k * 2^-24 of its terms'
            # size, so its rounding may fall one step apart. A normalised x one step apart in
            # one element moves y by ULP / sqrt(k) of one term, below that step. Through
            # SwiGLU: one step of each factor and two roundings.
            steps = 4 if kw.get("swiglu") else 2
            size = 1 + ref.abs() + (residual.float().abs() if "residual" in kw else 0)
            assert ((got - ref).abs() <= steps * ULP[dtype] * size).all(), (kw.keys(), n is None)
            # and on average no further than the rounding of y itself
            assert (got - ref).abs().mean() <= 0.1 * ULP[dtype]


def test_block_linear_of_no_terms(device):
    """K = 0: the product is 0, whatever the output's memory held."""
    say("block_linear K = 0")
    x, w = (torch.empty(n, 0, dtype=torch.bfloat16, device=device) for n in (3, 4096))
    norm = torch.empty(0, device=device)
    residual = torch.randn(3, 4096, device=device).to(torch.bfloat16)
    for n in (None, norm):
        for kw, want in ((dict(), torch.zeros_like(residual)), (dict(residual=residual), residual),
                         (dict(swiglu=True), torch.zeros_like(residual[:, :2048]))):
            stale = torch.full_like(want, 7.0)
            del stale  # the next allocation of this size
            got = ops.block_linear(x, w, norm_weight=n, eps=1e-6, **kw)
            assert torch.equal(got, want)


def test_block_linear_refuses_other_shapes(device):
    x = torch.zeros(17, 64, dtype=torch.bfloat16, device=device)
    w = torch.zeros(32, 64, dtype=torch.bfloat16, device=device)
    for args in ((x, w), (x[:4], w[:8]), (x[:4, :32].contiguous(), w[:, :32].contiguous()), (x[:4], w[:, :32]),
                 (x[:4].float(), w.float())):
        with pytest.raises(ValueError):
            ops.block_linear(*args)
    with pytest.raises(ValueError):
        ops.block_linear(x[:4], w, swiglu=True, residual=x[:4, :16].contiguous())
