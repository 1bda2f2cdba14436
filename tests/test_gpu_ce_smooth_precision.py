"""Label-smoothed cross-entropy in fp32: the rounding of the label's gradient against float64."""
import pytest
import torch

from trainscale_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("a", [0.05, 0.1, 0.2])
@pytest.mark.parametrize("V", [1000, 4099])  # whole vectors, and elements after the last one
def test_label_gradient_rounds_once(gpu, V, a):
    """p - a / V - (1 - a) lies in [0.5, 1) in magnitude: one rounding there is 2^-25, and 1 - a
    is kept beyond fp32. p itself carries the rounding of lse and of its product with log2(e),
    each half an ulp of a value below 16, and of the sum of V exponentials: under 2^-18 of p."""
    g = torch.Generator(device="cpu").manual_seed(V)
    N = 256
    x = torch.randn(N, V, generator=g)
    labels = torch.randint(0, V, (N,), generator=g)
    labels[0], labels[1] = V - 1, 0
    p = x.double().log_softmax(-1).exp().gather(1, labels[:, None])[:, 0]
    want = p - a / V - (1.0 - a)
    xd, ld, one = x.to(gpu), labels.to(gpu), torch.ones(1, device=gpu)
    _, _, grad = ops.ce_forward_backward(xd, V, ld, one, label_smoothing=a)
    _, lse = ops.ce_forward(xd, V, ld, label_smoothing=a)
    grad2 = torch.empty_like(xd)
    ops.ce_backward(xd, V, ld, lse, one, grad2, V, label_smoothing=a)
    for got in (grad, grad2):
        at = got.gather(1, ld[:, None])[:, 0].cpu().double()
        # 2^-28: a itself reaches the kernel as fp32
        assert ((at - want).abs() <= 2.0 ** -25 + 2.0 ** -28 + p * 2.0 ** -18).all()
