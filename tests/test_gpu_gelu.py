"""The erf-GELU of the GEMM epilogues, elementwise (s2_gelu), against float64:
max(x, 0) - |x| Q(|x|) with Q from Abramowitz & Stegun 7.1.26, whose error is
at most 0.75e-7 in Q, plus the fp32 roundings of its evaluation and of the
final fma; small inputs and the negative tail relative to the value; and the
limits at large |x|."""
import math

import pytest

from seedvr2_ncnn_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lo,hi", [(-1e-3, 1e-3), (-1.0, 1.0), (-6.0, 6.0), (-40.0, 40.0)])
def test_gelu_error(lo, hi):
    import torch
    x = torch.linspace(lo, hi, 400001, dtype=torch.float64, device="cuda").float()
    d = x.double()
    ref = 0.5 * d * torch.erfc(-d / math.sqrt(2.0))
    err = (capi.gelu(x).double() - ref).abs()
    # one ulp of the result is at most |ref| 2^-23
    assert (err - 2 ** -23 * ref.abs()).max().item() <= 3e-7
    # and relative to x: 1.5e-6 of Q near zero
    if hi <= 1.0:
        assert (err / d.abs().clamp_min(1e-30))[d != 0].max().item() <= 1.5e-6


@pytest.mark.parametrize("hi,std", [(0.1, None), (1.0, None), (None, 0.02), (None, 0.1)])
def test_gelu_small_inputs(hi, std):
    """The rms error relative to x: at most 0.75e-7 of the formula in Q, and 0.34e-7
    of about four fp32 roundings of values near 0.5 (2^-25 sqrt(4 / 3))."""
    import torch
    gen = torch.Generator(device="cuda").manual_seed(5)
    x = (torch.linspace(-hi, hi, 400001, dtype=torch.float64, device="cuda").float() if hi else
         std * torch.randn(400001, generator=gen, device="cuda"))
    x = x[x != 0]
    d = x.double()
    rel = (capi.gelu(x).double() - 0.5 * d * torch.erfc(-d / math.sqrt(2.0))) / d
    assert rel.square().mean().sqrt().item() <= 1.2e-7


def test_gelu_negative_tail():
    """The formula's own relative error grows to 1.03% over [-8, -6] (evaluated
    in float64); values there are below 1e-8."""
    import torch
    x = torch.linspace(-8, -6, 400001, dtype=torch.float64, device="cuda").float()
    d = x.double()
    ref = 0.5 * d * torch.erfc(-d / math.sqrt(2.0))
    assert ((capi.gelu(x).double() - ref) / ref).abs().max().item() <= 0.02


def test_gelu_limits():
    import torch
    # (at -13 the value, -8e-38, is still a normal fp32 number; at -15 it is zero)
    x = torch.tensor([0.0, 13.0, 1e4, 1e30, -15.0, -1e4, -1e30, float("nan")], device="cuda")
    y = capi.gelu(x)
    assert torch.equal(y[:4], x[:4])
    assert torch.equal(y[4:7], torch.zeros(3, device="cuda"))
    assert torch.isnan(y[7])
