"""The erf-GELU of the GEMM epilogues, elementwise (s2_gelu), against float64:
the polynomial's error (2.7e-7 at most, over the whole line) plus an ulp of the
hardware's 2^x and of the final fma, and the limits at large |x|."""
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


def test_gelu_limits():
    import torch
    x = torch.tensor([0.0, 13.0, 1e4, 1e30, -13.0, -1e4, -1e30, float("nan")], device="cuda")
    y = capi.gelu(x)
    assert torch.equal(y[:4], x[:4])
    assert torch.equal(y[4:7], torch.zeros(3, device="cuda"))
    assert torch.isnan(y[7])
