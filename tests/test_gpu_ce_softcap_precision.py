"""The softcapped logit z = c tanh(x / c) of fp32 logits against float64: the lse of a row of one
column is z itself. Its roundings are those of the quotient, of tanh and of the product by c,
half an ulp each (0.29 rms), which count up to twice where a binade ends below the result's, and
what v_exp_f32 leaves in tanh. A reciprocal of c rounded once would move every z the same way."""
import math

import numpy as np
import pytest
import torch

from trainscale_amd import ops

pytestmark = pytest.mark.gpu
N = 1 << 18


def softcapped(x, cap):
    """z by the forward kernel and by the one-pass one."""
    lab = torch.zeros(len(x), dtype=torch.long, device=x.device)
    one = torch.ones(1, device=x.device)
    x = x[:, None].contiguous()
    return (ops.ce_forward(x, 1, lab, -100, 0.0, cap)[1],
            ops.ce_forward_backward(x, 1, lab, one, 1.0, -100, 0.0, cap)[1])


@pytest.mark.parametrize("cap", [7.3, 15.0, 20.0, 30.0, 50.0])
@pytest.mark.parametrize("lo,hi", [(0.0, 0.2), (0.0, 0.75), (0.75, 1.5), (1.5, 4.0), (4.0, 9.0)])
def test_softcapped_logit(gpu, cap, lo, hi):
    c = float(np.float32(cap))
    g = torch.Generator(device=gpu).manual_seed(3)
    u = lo + (hi - lo) * torch.rand(N, generator=g, device=gpu, dtype=torch.float64)
    x = (c * u * torch.where(u * 1e6 % 2 < 1, 1.0, -1.0)).float()
    ref = c * torch.tanh(x.double() / c)
    ulp = 2.0 ** (ref.abs().log2().floor() - 23)
    for z in softcapped(x, cap):
        err = (z.double() - ref) / ulp
        # over the whole run of u the factors of 2 average to 1.1: 1.1 sqrt(3) 0.29 = 0.55
        assert err.pow(2).mean().sqrt() <= 0.60 and (err * ref.sign()).mean().abs() <= 0.1


@pytest.mark.parametrize("cap", [1e-40, 1e-38, 1e-20, 2.0, 1e20, 1e36])
def test_extreme_caps_and_logits(gpu, cap):
    c = float(np.float32(cap))
    x = torch.tensor([0.0, 1.0, -5.0, 1e5, -1e10, math.inf, -math.inf], device=gpu)
    ref = c * torch.tanh(x.double() / c)
    for z in softcapped(x, cap):
        # the quotient may be rounded to a denormal
        torch.testing.assert_close(z.double(), ref, rtol=2.0 ** -21, atol=2.0 ** -148 * max(c, 1.0))
    for z in softcapped(torch.full((3,), math.nan, device=gpu), cap):
        assert bool(z.isnan().all())
