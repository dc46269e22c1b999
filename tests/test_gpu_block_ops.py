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
