"""fp32 gradients of narrow rows against float64, as relative errors in the 2-norm.

dx = rstd (dy w - xhat c1) carries rstd's error (4.5e-8 rms, of a sum, a division, a square
root and another division) and two roundings of values spread over a binade (2.4e-8 each): the
product by rstd and the FMA, which takes dy w unrounded: 5.7e-8; a rounding of dy w would make
it 6.2e-8. dW sums rows of both signs: each of log2(slots) levels of a tree rounds a partial sum
once (a chain over n slots makes that error grow as sqrt(n) instead), after `steps` rows a slot."""
import pytest
import torch

from trainscale_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,dw_bound", [
    (64, 64, 1.1e-7), (44, 96, 1.05e-7), (1040, 80, 1.35e-7), (4096, 128, 1.7e-7),
    (5000, 12, 1.6e-7), (512, 4, 1.8e-7), (262144, 32, 2.4e-7), (300, 256, 1.1e-7)])
def test_fp32_gradients(gpu, rows, cols, dw_bound):
    sq = torch.zeros(2, dtype=torch.float64)
    for seed in range(6):
        g = torch.Generator(device=gpu).manual_seed(seed)
        x, dy = (torch.randn(rows, cols, generator=g, device=gpu) for _ in range(2))
        w = 1 + 0.1 * torch.randn(cols, generator=g, device=gpu)
        _, rstd = ops.rmsnorm_forward(x, cols, w, 1e-6)
        dx, dw = ops.rmsnorm_backward(dy, cols, x, cols, w, rstd, True)
        xd, d = x.double(), dy.double()
        r = (xd.pow(2).mean(1, keepdim=True) + 1e-6).rsqrt()
        xh, dxh = xd * r, d * w.double()
        ref = (r * (dxh - xh * (dxh * xh).mean(1, keepdim=True)), (d * xh).sum(0))
        for i, (got, want) in enumerate(zip((dx, dw), ref)):
            sq[i] += ((got.double() - want).norm() / want.norm()).item() ** 2 / 6
    err = sq.sqrt().tolist()
    if cols >= 64:
        assert err[0] <= 6.2e-8, err
    assert err[1] <= dw_bound, err
