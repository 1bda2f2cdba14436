"""Cross-entropy rows whose first vectors lie far from the rest of the row, in both schedules
and at every workgroup shape, against float64. A lane of the one-pass kernel sums its terms
against its first vector's maximum: lanes with low references must not overflow together, nor
may a lane whose reference lies far below the others' lose a large value."""
import pytest
import torch

from test_gpu_ce_ragged import check, rows_at
from trainscale_amd import ops

pytestmark = pytest.mark.gpu
BF, F32 = torch.bfloat16, torch.float32
SHAPES = [(BF, 1000), (BF, 1003), (BF, 4000), (BF, 8192), (BF, 20001), (BF, 50257),
          (BF, 131072), (torch.float16, 4099), (F32, 1000), (F32, 16389), (F32, 65536)]


def both(x, V, labels, dl, a=0.0):
    """(loss, lse, grad) of the one-pass and of the two-pass schedule."""
    yield ops.ce_forward_backward(x, V, labels, dl, 1.0, -100, 0.0, 0.0, a)
    loss, lse = ops.ce_forward(x, V, labels, -100, 0.0, 0.0, a)
    grad = torch.empty_like(x)
    ops.ce_backward(x, V, labels, lse, dl, grad, V, 1.0, -100, 0.0, 0.0, a)
    yield loss, lse, grad


@pytest.mark.parametrize("dtype,V", SHAPES)
@pytest.mark.parametrize("a", [0.0, 0.1])
def test_low_and_high_first_vectors(gpu, dtype, V, a):
    ve = 4 if dtype == F32 else 8
    leads = [t * ve for t in (64, 256, 512, 1024) if t * ve < V]  # first vectors, by workgroup
    rows = []
    for lead in leads:
        for low, high in ((-84.0, 0.0), (0.0, 84.0), (-40.0, 0.0), (float("-inf"), 0.0)):
            r = torch.full((V,), high)
            r[:lead] = low
            rows.append(r)
        r = torch.full((V,), -20.0)  # lane 0's reference far below, its second vector the maximum
        r[:ve], r[ve:2 * ve], r[lead] = -88.0, 0.0, 0.5
        rows.append(r)
    N = len(rows)
    for off in (0, 1):
        buf, x, labels = rows_at(N, V, V, off, dtype, gpu, V)
        x.copy_(torch.stack(rows))
        labels.fill_(V - 1)  # a finite logit in every row
        dl = torch.linspace(0.5, 0.9, N, device=gpu)
        if a:  # the smoothed loss of a row with -inf is inf
            x.clamp_(min=-1e4)
        for loss, lse, grad in both(x, V, labels, dl, a):
            check(grad, loss, x, labels, dl, a=a)
            torch.testing.assert_close(lse.double(), x.double().logsumexp(1), rtol=2.0 ** -22,
                                       atol=2.0 ** -18)


@pytest.mark.parametrize("dtype,V", SHAPES)
@pytest.mark.parametrize("cap", [0.0, 20.0])
def test_whole_vectors_of_nan(gpu, dtype, V, cap):
    """A row holding one vector of NaN only, or of NaN and -inf, in a lane's first vector or a
    later one, comes out NaN in both schedules; other rows do not."""
    ve = 4 if dtype == F32 else 8
    nvec = V // ve
    at = [0, 63, 64 % nvec, 255 % nvec, 300 % nvec, nvec - 1]
    N = 2 * len(at) + 1
    for off in (0, 1):
        buf, x, labels = rows_at(N, V, V, off, dtype, gpu, V)
        labels.fill_(V - 1)
        for i, v in enumerate(at):
            for r in (2 * i, 2 * i + 1):
                x[r, v * ve:(v + 1) * ve] = float("nan")
            if cap == 0.0:
                x[2 * i + 1, v * ve:v * ve + ve - 1] = float("-inf")
        dl = torch.ones(N, device=gpu)
        loss, lse, grad = ops.ce_forward_backward(x, V, labels, dl, 1.0, -100, 0.0, cap)
        loss2, lse2 = ops.ce_forward(x, V, labels, -100, 0.0, cap)
        for t in (loss, lse, loss2, lse2):
            assert bool(t[:-1].isnan().all()) and bool(t[-1:].isfinite().all())
        assert bool(grad[:-1].isnan().all()) and bool(grad[-1:].isfinite().all())


@pytest.mark.parametrize("dtype,V", SHAPES)
@pytest.mark.parametrize("low", ["lowest", -1e38, -1e9, 3e38])
def test_masked_with_the_lowest_value(gpu, dtype, V, low):
    """Logits at their type's lowest value, as masks leave them: in the first vectors, in one
    lane's, in all columns but one, in all columns; and logits near the largest."""
    low = torch.finfo(dtype).min if low == "lowest" else low
    if dtype == torch.float16 and abs(low) > 65504:
        pytest.skip("beyond fp16")
    ve = 4 if dtype == F32 else 8
    leads = [t * ve for t in (1, 64, 256, 512, 1024) if t * ve < V]
    N = len(leads) + 3
    for off in (0, 1):
        buf, x, labels = rows_at(N, V, V, off, dtype, gpu, V)
        labels.fill_(V - 1)
        for r, lead in enumerate(leads):
            x[r, :lead] = low
        x[N - 3, :V - 1] = low  # one column left
        x[N - 2, V // 2:V - 1] = low
        x[N - 1] = low  # nothing left: every logit is the maximum
        dl = torch.ones(N, device=gpu)
        if low > 0:  # the gradient needs lse * log2 e, which is past fp32 here
            lse = ops.ce_forward_backward(x, V, labels, dl)[1]
            for l in (lse, ops.ce_forward(x, V, labels)[1]):
                torch.testing.assert_close(l.double(), x.double().logsumexp(1), rtol=2.0 ** -23,
                                           atol=0)
            continue
        for loss, lse, grad in both(x, V, labels, dl):
            assert lse[N - 1] == x[N - 1, 0].float() + torch.tensor(float(V)).log()
            assert bool(loss[N - 1].isfinite())
            check(grad[:N - 1], loss[:N - 1], x[:N - 1], labels[:N - 1], dl[:N - 1])


@pytest.mark.parametrize("V", [1001, 4003, 16389, 65536])
@pytest.mark.parametrize("low", [0.0, -10.0, -20.0, -30.0, -40.0])
def test_lse_does_not_depend_on_the_reference(gpu, V, low):
    """lse to its own rounding wherever the lanes' first vectors lie. Its rms error in ulps: the
    last rounding (0.29); v_log_f32 and the lanes' own references, rounded at an ulp of 1 (0.15 of
    an lse between 4 and 8); v_exp_f32's ulp and the roundings of the sum and of exponents of up
    to 60, 2^-24 to 2^-20 a term, averaged over hundreds of them (0.1): together below 0.45."""
    for lead in (256, 1024, 2048, 4096):
        if lead > V // 2:
            break
        g = torch.Generator(device=gpu).manual_seed(V + lead)
        x = torch.randn(512, V, generator=g, device=gpu)
        x[:, :lead] += low
        labels = torch.zeros(512, dtype=torch.long, device=gpu)
        lse = ops.ce_forward_backward(x, V, labels, torch.ones(1, device=gpu))[1]
        ref = x.double().logsumexp(1)
        ulp = 2.0 ** (ref.log2().floor() - 23)
        err = (lse.double() - ref) / ulp
        assert err.pow(2).mean().sqrt().item() <= 0.45, (lead, err.pow(2).mean().sqrt().item())


@pytest.mark.parametrize("V", [1000, 1001, 4003])
@pytest.mark.parametrize("off", [160.0, -1000.0])
def test_lse_of_offset_logits(gpu, V, off):
    """With logits far from 0 on one side the sum's errors lie below an ulp of lse: what is left is
    its own rounding, sqrt(1 / 12) = 0.2887 ulp rms, and no bias, in both schedules."""
    g = torch.Generator(device=gpu).manual_seed(V)
    x = 2 * torch.randn(8192, V, generator=g, device=gpu) + off
    labels = torch.zeros(8192, dtype=torch.long, device=gpu)
    ref = x.double().logsumexp(1)
    ulp = 2.0 ** (ref.abs().log2().floor() - 23)
    one = torch.ones(1, device=gpu)
    for lse in (ops.ce_forward_backward(x, V, labels, one)[1], ops.ce_forward(x, V, labels)[1]):
        err = (lse.double() - ref) / ulp
        assert err.pow(2).mean().sqrt() <= 0.297 and err.mean().abs() <= 0.02
