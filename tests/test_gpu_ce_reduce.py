"""The row weight and the reduced loss formed by one workgroup, at the sizes where its loop
and the switch to torch's reductions turn, against float64. The weight is one fp32 division, the
loss a double sum divided in double and rounded once: half an fp32 ulp each."""
import pytest
import torch

from trainscale_amd import ops
from trainscale_amd.loss import FusedCrossEntropyLoss
from trainscale_amd.loss.sota_losses import _ONE_GROUP_ROWS, _hinted_weight, _reduced

pytestmark = pytest.mark.gpu
RED = ["mean", "sum", "batchmean"]


@pytest.mark.parametrize("n", [0, 1, 63, 1024, 8191, 8193, 16385, _ONE_GROUP_ROWS,
                               _ONE_GROUP_ROWS + 1])
@pytest.mark.parametrize("red", RED)
def test_weight_and_reduction(gpu, n, red):
    g = torch.Generator(device=gpu).manual_seed(n)
    labels = torch.randint(0, 50, (n,), generator=g, device=gpu)
    labels[::3] = 7
    rows = torch.rand(n, generator=g, device=gpu) * 20
    hint = torch.tensor([0.25], device=gpu)
    valid = int((labels != 7).sum())
    div = {"mean": max(valid, 1), "sum": 1, "batchmean": max(n, 1)}[red]
    w, used = _hinted_weight(labels, 7, red, n, hint)
    assert w.shape == (1,) and abs(w.item() * div - 0.25) <= 0.25 * 2.0 ** -23
    assert used.item() == 0.25 and used.data_ptr() != hint.data_ptr()
    w, used = _hinted_weight(labels, 7, red, n, None)
    assert used is None and abs(w.item() * div - 1.0) <= 2.0 ** -23
    loss = _reduced(rows, labels, 7, red)
    ref = rows.double().sum().item() / div
    # torch's own fp32 sum, taken above the switch, adds up to log2(n) roundings more
    tol = 2.0 ** -23 * (1 if n <= _ONE_GROUP_ROWS else 20)
    assert loss.shape == () and abs(loss.item() - ref) <= tol * abs(ref)


def test_all_ignored_and_int32_labels(gpu):
    logits = torch.randn(6, 40, device=gpu).requires_grad_()
    for labels in (torch.full((6,), -100, device=gpu), torch.arange(6, device=gpu).int()):
        loss = FusedCrossEntropyLoss()(logits, labels)
        ref = torch.nn.functional.cross_entropy(logits, labels.long(), reduction="sum")
        ref = ref / max(int((labels != -100).sum()), 1)
        torch.testing.assert_close(loss, ref.detach(), rtol=1e-6, atol=0)


def test_errors():
    import ctypes
    from trainscale_amd import _lib
    lib = _lib.load()
    null, fake = ctypes.c_void_p(0), ctypes.c_void_p(4096)
    invalid, shape = -1, -3
    assert lib.ts_ce_loss_weight(null, 4, -100, 0, null, fake, null, null) == invalid
    assert lib.ts_ce_loss_weight(fake, 4, -100, 0, null, null, null, null) == invalid
    assert lib.ts_ce_loss_weight(fake, 4, -100, 3, null, fake, null, null) == invalid
    assert lib.ts_ce_loss_weight(fake, -1, -100, 0, null, fake, null, null) == shape
    assert lib.ts_ce_reduce_loss(null, fake, 4, -100, 0, fake, null) == invalid
    assert lib.ts_ce_reduce_loss(fake, null, 4, -100, 0, fake, null) == invalid
    assert lib.ts_ce_reduce_loss(fake, fake, 4, -100, 0, null, null) == invalid
    assert lib.ts_ce_reduce_loss(fake, fake, 1 << 31, -100, 1, fake, null) == shape
