"""Default chunks of the linear-CE schedules: one token chunk while the bf16 logits fit in
1 GiB, vocabulary chunks as wide as 256 MB of dlogits allow. The rules on the CPU, and on the
GPU that the defaults are, bit for bit, the one-chunk calls they stand for."""
import pytest
import torch

from trainscale_amd import _lib
from trainscale_amd.loss import linear_ce as L

BF = torch.bfloat16


@pytest.mark.parametrize("N,V,rows", [(1, 8, 0), (512, 1000, 0), (1 << 16, 8, 0),
                                      (256, 1 << 22, 0), (4096, 1 << 17, 0),
                                      (4097, 1 << 17, 2304), (8192, 128256, 4096),
                                      (4099, (1 << 17) - 5, 2304), (300, 1 << 21, 256)])
def test_token_chunk(N, V, rows):
    assert L._chunk_rows(N, V, None) == rows
    assert L._chunk_rows(N, V, 512) == 512 and L._chunk_rows(N, V, 0) == 0


# dlogits bytes of the default chunk: the widest whole tiles within 256 MB, never fewer than
# V / 8 or 4096 columns, never past round_up(V, 8)
@pytest.mark.parametrize("N,V,cols", [(1, 50257, 50264), (1000, 32000, 32000),
                                      (2000, 128256, 67072), (8192, 128256, 16384),
                                      (65536, 128256, 16128), (65536, 20000, 4096),
                                      (1 << 28, 5000, 4096)])
def test_vocab_chunk_workspace(N, V, cols):
    lib = _lib.load()
    default = lib.ts_flce_backward_workspace_size(N, 64, V, 0)
    assert default == lib.ts_flce_backward_workspace_size(N, 64, V, cols)
    if cols > 256:
        assert default != lib.ts_flce_backward_workspace_size(N, 64, V, cols - 256)


@pytest.mark.gpu
@pytest.mark.parametrize("N,H,V", [(1, 8, 8), (300, 72, 9001), (777, 136, 20000)])
def test_defaults_are_one_chunk(gpu, N, H, V):
    g = torch.Generator(device=gpu).manual_seed(N + V)
    h = torch.randn(N, H, generator=g, device=gpu).to(BF)
    w = (0.05 * torch.randn(V, H, generator=g, device=gpu)).to(BF)
    labels = torch.randint(0, V, (N,), generator=g, device=gpu)
    a = L.linear_ce_forward_backward(h, w, labels)
    b = L.linear_ce_forward_backward(h, w, labels, chunk_tokens=0)
    assert all(torch.equal(x, y) for x, y in zip(a, b))
    lse = L.linear_ce_forward(h, w, labels)[2]
    one = torch.ones((), device=gpu)
    c = L.linear_ce_backward(h, w, labels, lse, one)
    d = L.linear_ce_backward(h, w, labels, lse, one, vocab_chunk=V)
    assert all(torch.equal(x, y) for x, y in zip(c, d))
    assert torch.equal(a[3], c[0]) and torch.equal(a[4], c[1])
