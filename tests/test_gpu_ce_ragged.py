"""Cross-entropy rows at every address phase and workgroup shape, with and without smoothing
and transforms, against float64.

The bound of a gradient element is derived: with p = exp(z - lse) formed as
exp2(fma(z, log2 e, -lse log2 e)), the exponent carries an absolute error of about
(|z| + |lse|) 2^-23 (its rounding and that of lse), softcapping adds 2 ulps of z, and
1 - tanh^2 one of 2^-22; the label's and the smoothing's terms are rounded once each, and the
result once to its type."""
import pytest
import torch

from trainscale_amd import ops

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
HALF_ULP = {BF: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}
# v_exp_f32 flushes results below the smallest normal fp32 value (2^-126) to zero
TINY = {BF: 2.0 ** -125, torch.float16: 2.0 ** -24, torch.float32: 2.0 ** -125}


def rows_at(N, V, ld, off, dtype, dev, seed):
    """[N, V] logits whose first row starts `off` elements into a 16-byte aligned buffer."""
    g = torch.Generator(device=dev).manual_seed(seed)
    buf = (3 * torch.randn(off + N * ld, generator=g, device=dev)).to(dtype)
    labels = torch.randint(0, V, (N,), generator=g, device=dev)
    labels[0], labels[N - 1] = 0, V - 1  # labels in the ragged ends
    labels[1] = -100
    return buf, buf[off:].as_strided((N, V), (ld, 1)), labels


def reference(x, labels, dl, sc=0.0, cap=0.0, a=0.0):
    """(loss, lse, grad, bound of grad) in float64."""
    V = x.shape[1]
    s = sc if sc != 0.0 else 1.0
    z, dz = x.double() * s, torch.full_like(x.double(), s)
    if cap:
        t = torch.tanh(z / cap)
        z, dz = cap * t, (1 - t * t) * s
    ok = labels != -100
    lab = labels.clamp(min=0)[:, None]
    lse = z.logsumexp(1)
    zt = z.gather(1, lab)[:, 0]
    loss = (1 - a) * (lse - zt) * ok
    if a:
        loss = loss + a * (lse - z.mean(1)) * ok
    p = (z - lse[:, None]).exp()
    hot = torch.zeros_like(p).scatter_(1, lab, 1.0)
    up = (dl.double() * ok)[:, None]
    grad = up * (p - (1 - a) * hot - a / V) * dz
    u = 2.0 ** -23
    size = torch.where(z.isinf(), torch.zeros_like(z), z.abs())  # p is 0 at -inf
    err = u * (8 + 4 * size + 2 * lse.abs()[:, None]) * p + 2 * u * (hot + a / V)
    b = up.abs() * (err * dz.abs() + (4 * u * abs(s) * (p + hot + a / V) if cap else 0.0))
    return loss, lse, grad, b


def check(got, loss, x, labels, dl, **kw):
    ref_loss, lse, ref, b = reference(x, labels, dl, **kw)
    tol = 1e-5 * ref_loss.abs() + 4 * 2.0 ** -23 * lse.abs().clamp(min=1)
    assert bool(((loss.double() - ref_loss).abs() <= tol).all())
    b = b + HALF_ULP[got.dtype] * (ref.abs() + b) + TINY[got.dtype]
    bad = (got.double() - ref).abs() > b
    assert not bool(bad.any()), (bad.nonzero()[:4].tolist(), int(bad.sum()))


# around the row lengths where the shape changes (8 bf16 or 4 fp32 values a vector), and rows
# with no aligned vector at all
@pytest.mark.parametrize("dtype,V", [(BF, 1), (BF, 6), (BF, 8), (BF, 15), (BF, 8191), (BF, 8200),
                                     (BF, 16383), (BF, 16392), (BF, 32769), (BF, 50257),
                                     (BF, 65543), (BF, 131071), (BF, 131081),
                                     (torch.float16, 4099), (torch.float32, 3),
                                     (torch.float32, 16389), (torch.float32, 32773)])
@pytest.mark.parametrize("kw", [dict(), dict(a=0.1), dict(sc=0.5, cap=20.0), dict(sc=-1.5),
                                dict(cap=2.0, a=0.2)])
def test_one_pass_and_two_pass(gpu, dtype, V, kw):
    N = 5
    ve = 4 if dtype == torch.float32 else 8
    for off, pad in ((0, 0), (3 % ve, 0), (1, 5)):
        buf, x, labels = rows_at(N, V, V + pad, off, dtype, gpu, V + off)
        dl = torch.linspace(-0.7, 0.9, N, device=gpu)
        args = (-100, kw.get("sc", 0.0), kw.get("cap", 0.0), kw.get("a", 0.0))
        # logits at one phase, the gradient packed (another) or laid out like the logits;
        # the results do not depend on either
        same = torch.full_like(buf, float("nan"))[off:].as_strided((N, V), (V + pad, 1))
        loss, lse, packed = ops.ce_forward_backward(x, V + pad, labels, dl, 1.0, *args)
        check(packed, loss, x, labels, dl, **kw)
        again = ops.ce_forward_backward(x.contiguous(), V, labels, dl, 1.0, *args)
        assert all(torch.equal(p, q) for p, q in zip((loss, lse, packed), again))
        loss2, lse2 = ops.ce_forward(x, V + pad, labels, *args)
        ops.ce_backward(x, V + pad, labels, lse2, dl, same, V + pad, 1.0, *args)
        check(same, loss2, x, labels, dl, **kw)
        other = torch.full((N, V), float("nan"), dtype=dtype, device=gpu)
        ops.ce_backward(x, V + pad, labels, lse2, dl, other, V, 1.0, *args)
        assert torch.equal(other, same)
        # in place over the logits; what lies around the rows stays
        keep = buf.clone()
        ops.ce_backward(x, V + pad, labels, lse2, dl, x, V + pad, 1.0, *args)
        assert torch.equal(x, same)
        inside = torch.zeros_like(buf, dtype=torch.bool)
        inside[off:].as_strided((N, V), (V + pad, 1)).fill_(True)
        assert torch.equal(buf[~inside], keep[~inside])


@pytest.mark.parametrize("V", [50257, 777])
def test_extreme_ragged_ends(gpu, V):
    """-inf, the row's maximum and NaN in the first elements and in those after the last
    whole vector."""
    buf, x, labels = rows_at(6, V, V, 3, BF, gpu, 1)
    x[0, :5], x[2, :9] = float("-inf"), 90.0
    x[3, V - 2:] = 95.0
    x[4, 0] = float("nan")
    x[5] = float("-inf")
    x[5, V - 1] = 1.0
    labels[0] = 9
    labels[4] = 7
    dl = torch.ones(6, device=gpu)
    loss, lse, grad = ops.ce_forward_backward(x.contiguous(), V, labels, dl)
    loss2, _ = ops.ce_forward(x, V, labels)
    fine = torch.tensor([True, True, True, True, False, True], device=gpu)
    ref_loss, _, ref, b = reference(x[fine], labels[fine], dl[fine])
    assert bool(loss[4].isnan()) and bool(grad[4].isnan().all()) and bool(loss2[4].isnan())
    for l in (loss[fine], loss2[fine]):
        torch.testing.assert_close(l.double(), ref_loss, rtol=1e-5, atol=1e-4)
    b = b + 2.0 ** -8 * (ref.abs() + b) + TINY[BF]
    assert bool(((grad[fine].double() - ref).abs() <= b).all())
