"""grad_hidden summed over K slots (ts_plan::hidden_split) on the GPU: every element within
the bound of a K = V GEMM (tests/lce_bounds.py; a sum of slots adds at most one fp32 rounding
of the partial per slot, which the bound's K / 16 roundings exceed), the three schedules bit
for bit alike where they sum the same K, and last chunks so short that slots stay empty."""
import pytest
import torch

from test_gpu_linear_ce import _token_chunk, _vocab_chunks, check_grads, make_ref

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _inputs(N, H, V, dev):
    g = torch.Generator(device=dev).manual_seed(N + H + V)
    h = torch.randn(N, H, generator=g, device=dev).to(BF)
    w = (0.05 * torch.randn(V, H, generator=g, device=dev)).to(BF)
    labels = torch.randint(0, V, (N,), generator=g, device=dev)
    labels[::11] = -100
    return h, w, labels


# V: just split into 2 slots, an odd one with a short last slot, one with many slots
@pytest.mark.parametrize("N,H,V", [(200, 136, 4096), (257, 72, 9001), (520, 264, 12345)])
def test_schedules_agree_when_split(gpu, N, H, V):
    from trainscale_amd.loss.linear_ce import (linear_ce_backward, linear_ce_forward,
                                               linear_ce_forward_backward)
    h, w, labels = _inputs(N, H, V, gpu)
    ref = make_ref(h, w, labels)  # the stored-logits gradients, checked on the way
    _, _, lse, gh1, gw1 = linear_ce_forward_backward(h, w, labels, chunk_tokens=0)
    check_grads(gh1, gw1, ref, what="one call")
    one = torch.ones((), device=gpu)
    _, _, lse2 = linear_ce_forward(h, w, labels)
    gh2, gw2 = linear_ce_backward(h, w, labels, lse2, one, vocab_chunk=V)
    assert torch.equal(gh1, gh2) and torch.equal(gw1, gw2)
    _, _, lse3, logits = linear_ce_forward(h, w, labels, keep_logits=True)
    gh3, gw3 = linear_ce_backward(h, w, labels, lse3, one, logits=logits)
    assert torch.equal(gh1, gh3) and torch.equal(gw1, gw3)
    # grad_hidden alone (no grad_weight in the grid) is the same sum
    gh4, none = linear_ce_backward(h, w, labels, lse2, one, vocab_chunk=V, need_grad_weight=False)
    assert none is None and torch.equal(gh1, gh4)


# two-pass chunks of 4096 columns (2 slots) whose last chunk is short, or leaves a slot empty
@pytest.mark.parametrize("N,H,V", [(200, 136, 4096 + 808), (130, 264, 2 * 4096 + 8)])
def test_two_pass_chunks_with_slots(gpu, N, H, V):
    from trainscale_amd.loss.linear_ce import linear_ce_backward, linear_ce_forward
    h, w, labels = _inputs(N, H, V, gpu)
    ref = make_ref(h, w, labels)
    _, _, lse = linear_ce_forward(h, w, labels)
    gh, gw = linear_ce_backward(h, w, labels, lse, torch.ones((), device=gpu), vocab_chunk=4096)
    check_grads(gh, gw, ref, vocab_chunks=_vocab_chunks(V, 4096), what="two-pass slots")


def test_token_chunks_with_slots(gpu):
    """Token chunks of different row counts (512, then 88: cut into more slots)."""
    from trainscale_amd.loss.linear_ce import linear_ce_forward_backward
    N, H, V = 600, 264, 20000
    h, w, labels = _inputs(N, H, V, gpu)
    tc = _token_chunk(N, V, 512)
    ref = make_ref(h, w, labels, token_chunk=tc)
    for accum, mode in (("bf16", "bf16_run"), ("fp32", "f32_run")):
        _, _, _, gh, gw = linear_ce_forward_backward(h, w, labels, chunk_tokens=512,
                                                     grad_weight_accum=accum)
        check_grads(gh, gw, ref, gw_mode=mode, what=f"token chunks {accum}")
