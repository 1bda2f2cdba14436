"""Partials of a vocabulary shard whose first vectors lie far from the rest, hold NaN or are
masked with the type's lowest value, at every register shape, against float64."""
import pytest
import torch

from trainscale_amd import ops

pytestmark = pytest.mark.gpu
BF, F32 = torch.bfloat16, torch.float32
SHAPES = [(BF, 2048), (BF, 2056), (BF, 8192), (BF, 16032), (BF, 32768), (BF, 50264),
          (torch.float16, 6144), (F32, 4096), (F32, 65536)]


def stats_of(rows, dtype, dev, nan=0):
    x = torch.stack(rows).to(dtype).to(dev)
    t = torch.zeros(len(rows), dtype=torch.long, device=dev)
    stats = ops.ce_vocab_shard_stats(x, x.shape[1], t, 0)
    return x, stats[:, 0], ops.ce_vocab_merge(stats[None], 0, x.shape[1])[0]


@pytest.mark.parametrize("dtype,V", SHAPES)
def test_far_references(gpu, dtype, V):
    ve = 4 if dtype == F32 else 8
    low = torch.finfo(dtype).min
    rows = []
    for lead in (t * ve for t in (1, 256, 512, 1024) if t * ve < V):
        for a, b in ((-84.0, 0.0), (0.0, 84.0), (-40.0, 0.0), (low, 0.0), (-1e9, 1.0),
                     (float("-inf"), 0.0)):
            r = torch.full((V,), b)
            r[:lead] = max(a, low) if a != float("-inf") else a
            rows.append(r)
        r = torch.full((V,), -20.0)  # a low reference over the row's maximum
        r[:ve], r[ve:2 * ve], r[lead] = -88.0, 0.0, 0.5
        rows.append(r)
    x, lse, merged = stats_of(rows, dtype, gpu)
    # lse to a few roundings of its own size (the merge of one rank keeps it)
    ref = x.double().logsumexp(1)
    for l in (lse, merged):
        torch.testing.assert_close(l.double(), ref, rtol=2.0 ** -22, atol=2.0 ** -21)


@pytest.mark.parametrize("dtype,V", SHAPES)
def test_vectors_of_nan(gpu, dtype, V):
    ve = 4 if dtype == F32 else 8
    rows = []
    for v in (0, 63, 255, 300 % (V // ve), V // ve - 1):
        r = torch.zeros(V)
        r[v * ve:(v + 1) * ve] = float("nan")
        rows.append(r)
    rows.append(torch.full((V,), float("nan")))
    _, lse, merged = stats_of(rows, dtype, gpu)
    assert bool(lse.isnan().all()) and bool(merged.isnan().all())
